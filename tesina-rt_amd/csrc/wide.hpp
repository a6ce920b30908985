// Wide records: the four-wide form of the BVH that groups of four lanes walk.
//
// A wide record holds the (up to) four grandchildren of an inner node: the
// children of its left child, or the left child itself when that is a leaf,
// then the same for the right child.  Four slots of 32 bytes, one 128-byte
// line: {lo.xyz, ref | hi.xyz, 0}.  The record of an inner node with left
// child a (odd) is number (a - 1) / 2, so a record needs no index of its own;
// only the nodes at even levels have one written.
//
// ref is what the walk pushes on its stack:
//   inner node: its record's number, WIDE_DEEP set where the reference's
//     MAX_LEVELS rule can show below it (an inner child at level 31);
//   leaf: WIDE_LEAF, the triangle count (1..15) in bits 27..30 and the first
//     triangle; for larger leaves the count bits are 0 and the rest is the
//     leaf's node number;
//   WIDE_EMPTY: no child (the second slot of a leaf child).
#pragma once

#include "devmath.hpp"
#include "rtx_impl.hpp"

constexpr uint32_t WIDE_EMPTY = 0xffffffffu;
constexpr uint32_t WIDE_LEAF = 0x80000000u, WIDE_DEEP = 0x10000000u, WIDE_LOW = 0x07ffffffu;
// Most triangles of a tree with wide records (27-bit references; record
// offsets in 32 bits).
constexpr uint32_t WIDE_MAX_TRIS = 1u << 25;
// Stack entries per ray.  A step replaces one entry by at most four, so 49
// would hold any walk above level 30; rays that need more than these are
// walked node by node.  With 32, a wave of the closest-hit walk takes 4.3 KB of
// LDS where a group holds its ray (7 waves per SIMD, by registers) and 8 KB
// where 64 rays wait in LDS (5 waves per SIMD, by LDS).
constexpr int WIDE_STACK = 32;

__device__ __forceinline__ uint32_t wide_ref(uint32_t n, uint32_t a, uint32_t cnt) {
    if (cnt == 0u) return (a - 1u) >> 1;
    return WIDE_LEAF | (cnt <= 15u ? (cnt << 27) | a : n);
}

// Leaves tested by the whole wave in the wide walk: four times the size of the
// single-lane forms' (a group tests four triangles at a time).
inline uint32_t rtx_wide_coop(const rtx_ctx* c) {
    return c->tune.coop_leaf > 0 ? 4u * (uint32_t)c->tune.coop_leaf : 0xffffffffu;
}
