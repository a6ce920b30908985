// LBVH build on gfx950: prim AABB + global AABB, Morton codes, onesweep
// radix sort, permutation of the scene buffers, every node of the level-ordered
// hierarchy from its split, boxes by unions over the sorted positions, and the
// child pairs' differences and wide records.
//
// Reference: BVHBuilder::build_lbvh / refit_lbvh (src/rt/bvh-builder.cpp:201-850)
// with the kernels of src/kernel/bvh-builder.cl and bvh-builder-sort.cl.
//
// Result contract (checked against the oracle): identical Morton codes,
// the permutation of a stable sort by (code, input position), nodes in
// canonical level order (root, then each iteration's children block ordered
// by parent position, left before right — what process_task produces when
// its work-groups run in order), identical node AABBs.
#include <cstring>

#include "devmath.hpp"
#include "lookback.hpp"
#include "rtx_impl.hpp"
#include "wide.hpp"

namespace {

constexpr int BS = 256;
constexpr int SORT_ITEMS = 16;               // the smallest tile (sizes the look-back words)
constexpr int SORT_TILE = BS * SORT_ITEMS;
constexpr int BOUNDS_GRID = 512;
constexpr int TREE_TILE = 1024;              // tree phase: sorted positions per tile
constexpr uint32_t NONE = 0xffffffffu;

// Counter slots in scene->tickets.
constexpr int TK_BOUNDS = 0;
constexpr int TK_SORT = 1;    // up to 8 passes (4-bit digits)
constexpr int TK_RANK = 16;
constexpr int TK_COUNT = 80;

// Layout of scene->levels (uint32): [d] = first node of level d,
// [64 + d] = node count of level d, [128] = total node count.
constexpr int LV_OFF = 0, LV_CNT = 64, LV_TOTAL = BuildSet::NODE_COUNT, LV_WORDS = 192;

// ------------------------------------------------------------- helpers --
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x, uint32_t lane) {
    for (int off = 1; off < RTX_WAVE; off <<= 1) {
        uint32_t y = __shfl_up(x, off, RTX_WAVE);
        if (lane >= (uint32_t)off) x += y;
    }
    return x;
}

// Exclusive scan of one value per thread over a block of NT threads.
template <int NT = BS>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t x, uint32_t* s_w, uint32_t* total) {
    uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = wave_incl_scan(x, lane);
    if (lane == 63) s_w[w] = inc;
    __syncthreads();
    uint32_t base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NT / RTX_WAVE; ++i) {
        uint32_t v = s_w[i];
        base += (i < (int)w) ? v : 0u;
        tot += v;
    }
    __syncthreads();
    *total = tot;
    return base + inc - x;
}

// -------------------------------------------------------------- kernels --
__global__ __launch_bounds__(BS) void k_build_init(uint32_t* zero_a, uint32_t na, uint32_t* zero_b, uint32_t nb,
                                                   uint32_t* zero_c, uint32_t nc, uint32_t* zero_d, uint32_t nd,
                                                   uint32_t* levels, uint32_t* parent) {
    uint32_t stride = gridDim.x * BS;
    for (uint32_t i = blockIdx.x * BS + threadIdx.x; i < na; i += stride) zero_a[i] = 0;
    for (uint32_t i = blockIdx.x * BS + threadIdx.x; i < nb; i += stride) zero_b[i] = 0;
    for (uint32_t i = blockIdx.x * BS + threadIdx.x; i < nc; i += stride) zero_c[i] = 0;
    for (uint32_t i = blockIdx.x * BS + threadIdx.x; i < nd; i += stride) zero_d[i] = 0;
    if (blockIdx.x == 0) {
        // every word is written once, by one thread, with its final value:
        // the root's count and the node total are 1, the rest 0 (a zeroing
        // pass followed by a store of the root words from another wave would
        // race with it)
        for (uint32_t i = threadIdx.x; i < LV_WORDS; i += BS)
            levels[i] = (i == (uint32_t)(LV_CNT + 0) || i == (uint32_t)LV_TOTAL) ? 1u : 0u;
        if (threadIdx.x == 0) parent[0] = 0;
    }
}

// build_primitive_bbox + max_local_bbox (src/kernel/bvh-builder.cl:100-130,
// 318-391): per-triangle AABB, its centroid (hi+lo)*0.5 for the Morton
// stage, and the union of all AABBs (last block to finish reduces the
// per-block partials).
__global__ __launch_bounds__(BS) void k_prim_bounds(const uint32_t* __restrict__ idx, const float4* __restrict__ pos,
                                                    float4* __restrict__ cen, float* __restrict__ partials,
                                                    uint32_t T) {
    __shared__ float s_r[6][BS / RTX_WAVE];
    v3 lo = mk3(INFINITY, INFINITY, INFINITY), hi = mk3(-INFINITY, -INFINITY, -INFINITY);
    for (uint32_t i = blockIdx.x * BS + threadIdx.x; i < T; i += gridDim.x * BS) {
        uint32_t i0 = idx[3 * (size_t)i], i1 = idx[3 * (size_t)i + 1], i2 = idx[3 * (size_t)i + 2];
        v3 v0 = xyz(pos[i0]), v1 = xyz(pos[i1]), v2 = xyz(pos[i2]);
        v3 bhi = v0, blo = v0;
        bhi = vmax(bhi, v1);
        bhi = vmax(bhi, v2);
        blo = vmin(blo, v1);
        blo = vmin(blo, v2);
        v3 c = (bhi + blo) * 0.5f;
        cen[i] = make_float4(c.x, c.y, c.z, 0.f);
        lo = vmin(lo, blo);
        hi = vmax(hi, bhi);
    }
    float r[6] = {lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) r[k] = fminf(r[k], __shfl_xor(r[k], off, RTX_WAVE));
#pragma unroll
        for (int k = 3; k < 6; ++k) r[k] = fmaxf(r[k], __shfl_xor(r[k], off, RTX_WAVE));
    }
    uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0)
        for (int k = 0; k < 6; ++k) s_r[k][w] = r[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int ww = 1; ww < BS / RTX_WAVE; ++ww) {
            for (int k = 0; k < 3; ++k) r[k] = fminf(r[k], s_r[k][ww]);
            for (int k = 3; k < 6; ++k) r[k] = fmaxf(r[k], s_r[k][ww]);
        }
        for (int k = 0; k < 6; ++k) partials[6 * blockIdx.x + k] = r[k];
    }
}

// Union of the per-block partial AABBs (one block).
__global__ __launch_bounds__(BS) void k_gbox_reduce(const float* __restrict__ partials, uint32_t nparts,
                                                    float* __restrict__ gbox6) {
    __shared__ float s_r[6][BS / RTX_WAVE];
    float q[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (uint32_t b = threadIdx.x; b < nparts; b += BS) {
        for (int k = 0; k < 3; ++k) q[k] = fminf(q[k], partials[6 * b + k]);
        for (int k = 3; k < 6; ++k) q[k] = fmaxf(q[k], partials[6 * b + k]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) q[k] = fminf(q[k], __shfl_xor(q[k], off, RTX_WAVE));
#pragma unroll
        for (int k = 3; k < 6; ++k) q[k] = fmaxf(q[k], __shfl_xor(q[k], off, RTX_WAVE));
    }
    uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0)
        for (int k = 0; k < 6; ++k) s_r[k][w] = q[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int ww = 1; ww < BS / RTX_WAVE; ++ww) {
            for (int k = 0; k < 3; ++k) q[k] = fminf(q[k], s_r[k][ww]);
            for (int k = 3; k < 6; ++k) q[k] = fmaxf(q[k], s_r[k][ww]);
        }
        for (int k = 0; k < 6; ++k) gbox6[k] = q[k];
    }
}

// morton_encode (src/kernel/bvh-builder.cl:181-252): centroid normalized to
// the global AABB with a reciprocal then a multiply, clamped with
// fmax(0, fmin(1, s)), scaled by 2^ceil(depth/3), truncated; bit i of the
// code takes axis (off+1+i)%3, source bit (i+off)/3.  Also accumulates the
// 8-bit digit histograms of every radix pass.
// Bit k of v (k < 11) to bit 3k.
__device__ __forceinline__ uint64_t spread3(uint32_t v) {
    uint64_t x = v & 0x7ffu;
    x = (x | (x << 16)) & 0x00000000ff0000ffull;
    x = (x | (x << 8)) & 0x000000f00f00f00full;
    x = (x | (x << 4)) & 0x00000c30c30c30c3ull;
    x = (x | (x << 2)) & 0x0000249249249249ull;
    return x;
}

__global__ __launch_bounds__(BS) void k_morton(const float4* __restrict__ cen, const float* __restrict__ gbox6,
                                               uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                               uint32_t* __restrict__ hist, uint32_t T, int depth, int passes,
                                               int rbits) {
    // digit histograms of every pass: pass p, digit d at p * 2^rbits + d
    // (4 passes of 8 bits or 8 of 4 bits: at most 1024 words)
    __shared__ uint32_t s_h[1024];
    for (int i = threadIdx.x; i < 1024; i += BS) s_h[i] = 0;
    __syncthreads();
    const uint32_t rmask = (1u << rbits) - 1u;
    v3 glo = mk3(gbox6[0], gbox6[1], gbox6[2]);
    v3 ghi = mk3(gbox6[3], gbox6[4], gbox6[5]);
    v3 inv = recip(ghi - glo);
    float scale = (float)(1u << ((depth + 2) / 3));
    const int offset = depth % 3 ? 3 - (depth % 3) : 0;
    const uint64_t dmask = depth >= 64 ? ~0ull : ((1ull << depth) - 1ull);
    const uint32_t lane = threadIdx.x & 63u;
    // all lanes of a wave step together (the histogram is aggregated per wave)
    for (uint32_t base = blockIdx.x * BS; base < T; base += gridDim.x * BS) {
        const uint32_t i = base + threadIdx.x;
        const bool active = i < T;
        uint32_t code = 0;
        if (active) {
            v3 c = xyz(cen[i]);
            v3 sl = (c - glo) * inv;
            sl = vmax(mk3(0.f, 0.f, 0.f), vmin(mk3(1.f, 1.f, 1.f), sl));
            sl = sl * scale;
            // bit b of the code is bit (b + offset) / 3 of axis (offset + 1 + b) % 3:
            // interleave y, z, x at bits 3k, 3k + 1, 3k + 2, shift by offset, keep depth bits
            const uint64_t f = spread3((uint32_t)sl.y) | (spread3((uint32_t)sl.z) << 1) |
                               (spread3((uint32_t)sl.x) << 2);
            code = (uint32_t)((f >> offset) & dmask);
            keys[i] = code;
            vals[i] = i;
        }
        const uint64_t act = ballot(active);
        const uint32_t lead = (uint32_t)__builtin_ctzll(act);
        for (int p = 0; p < passes; ++p) {
            const uint32_t d = (code >> (rbits * p)) & rmask;
            const uint32_t d0 = __shfl(d, (int)lead, RTX_WAVE);
            // input in the last build's order is nearly sorted: whole waves share a digit
            if (ballot(active && d == d0) == act) {
                if (lane == lead) atomicAdd(&s_h[(p << rbits) + d0], (uint32_t)__builtin_popcountll(act));
            } else if (active) {
                atomicAdd(&s_h[(p << rbits) + d], 1u);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < (passes << rbits); i += BS) {
        const uint32_t c = s_h[i];
        if (c) atomicAdd(&hist[i], c);
    }
}

// One stable LSD pass over `bits` <= RB bits at `shift` (onesweep: in-tile
// rank by wave64 ballot matching, per-digit decoupled look-back across tiles,
// LDS-staged scatter) over tiles of NT * ITEMS pairs.  Replaces the bitonic
// network of src/kernel/bvh-builder-sort.cl:26-232.  RB = 8: 256 digits a
// pass; RB = 4: 16 digits, twice the passes, longer runs per digit in the
// scatter (the reference's radix prototype, src/kernel/sort.cl:491-628, uses
// 4-bit digits).  The look-back word of tile t, digit d is status[t * 2^RB + d].
// A pass over few tiles is bound by one tile's latency (loads, ITEMS rank
// rounds, scans, look-back), so such tiles are spread over 1024 threads of 4
// pairs instead of 256 of 16: 13.1 to 9.9 us a pass over 65k pairs, 15.3 to
// 11.8 over 300k, 20.8 to 17.7 over 1M.  Over 2000 tiles the fewer, larger
// blocks per CU lose: 70 against 85 us at 8M.
template <int RB, int ITEMS, int NT>
__global__ __launch_bounds__(NT) void k_sort_pass(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                  uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                  uint32_t n, int shift, int bits, const uint32_t* __restrict__ hist,
                                                  uint32_t* status, uint32_t* ticket) {
    constexpr int TILE = NT * ITEMS;
    constexpr uint32_t DIG = 1u << RB;
    static_assert(DIG <= (uint32_t)NT, "one thread per digit");
    __shared__ uint32_t s_keys[TILE];
    __shared__ uint32_t s_vals[TILE];
    __shared__ uint32_t s_wcnt[NT / RTX_WAVE][DIG];
    __shared__ uint32_t s_tofs[DIG];
    __shared__ uint32_t s_gofs[DIG];
    __shared__ uint32_t s_w[NT / RTX_WAVE];
    __shared__ uint32_t s_tile;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (tid == 0) s_tile = atomicAdd(ticket, 1u);
    if (tid < DIG) {
#pragma unroll
        for (int i = 0; i < NT / RTX_WAVE; ++i) s_wcnt[i][tid] = 0;
    }
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t base = tile * TILE;
    const uint32_t dmask = (1u << bits) - 1u;

    uint32_t k[ITEMS], v[ITEMS], r[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        uint32_t e = base + (w * ITEMS + j) * RTX_WAVE + lane;
        bool ok = e < n;
        k[j] = ok ? kin[e] : 0xffffffffu;
        v[j] = ok ? vin[e] : 0u;
    }
    // global start of each digit = exclusive scan of the pass histogram
    uint32_t dummy;
    const uint32_t hv = tid <= dmask ? hist[tid] : 0u;
    const uint32_t dbase = block_excl_scan<NT>(hv, s_w, &dummy);
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        uint32_t e = base + (w * ITEMS + j) * RTX_WAVE + lane;
        bool ok = e < n;
        uint32_t d = (k[j] >> shift) & dmask;
        uint64_t peers = ballot(ok);
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            if (b < bits) {
                bool bit = (d >> b) & 1u;
                uint64_t bal = ballot(bit);
                peers &= bit ? bal : ~bal;
            }
        }
        uint32_t below = lanes_below(peers);
        uint32_t cnt = (uint32_t)__builtin_popcountll(peers);
        uint32_t basec = ok ? s_wcnt[w][d] : 0u;
        r[j] = basec + below;
        if (ok && below == 0) s_wcnt[w][d] = basec + cnt;
    }
    __syncthreads();
    // per-digit tile totals, wave offsets (exclusive, in wave order)
    uint32_t tot = 0;
    if (tid < DIG) {
        uint32_t c[NT / RTX_WAVE];
#pragma unroll
        for (int i = 0; i < NT / RTX_WAVE; ++i) c[i] = s_wcnt[i][tid];
#pragma unroll
        for (int i = 0; i < NT / RTX_WAVE; ++i) {
            s_wcnt[i][tid] = tot;
            tot += c[i];
        }
    }
    // successors can go on with this tile's counts before the scan below
    if (tid <= dmask) st_relaxed(&status[(size_t)tile * DIG + tid], (tile ? RTX_LB_AGG : RTX_LB_INC) | tot);
    uint32_t tofs = block_excl_scan<NT>(tot, s_w, &dummy);
    if (tid < DIG) s_tofs[tid] = tofs;
    if (tid <= dmask) {
        uint32_t prefix = lookback_thread(status + tid, tile, tot, DIG);
        s_gofs[tid] = dbase + prefix - tofs;  // dest = s_gofs[d] + local position
    }
    __syncthreads();
    // stage the tile in LDS in sorted order
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        uint32_t e = base + (w * ITEMS + j) * RTX_WAVE + lane;
        if (e < n) {
            uint32_t d = (k[j] >> shift) & dmask;
            uint32_t lp = s_tofs[d] + s_wcnt[w][d] + r[j];
            s_keys[lp] = k[j];
            s_vals[lp] = v[j];
        }
    }
    __syncthreads();
    uint32_t nvalid = n - base < (uint32_t)TILE ? n - base : (uint32_t)TILE;
    for (uint32_t i = tid; i < nvalid; i += NT) {
        uint32_t key = s_keys[i];
        uint32_t dst = s_gofs[(key >> shift) & dmask] + i;
        kout[dst] = key;
        vout[dst] = s_vals[i];
    }
}

// Copy of the buffers the build permutes in place (the reference copies each
// to an aux buffer first, src/rt/bvh-builder.cpp:481-527).
__global__ __launch_bounds__(BS) void k_stage_copy(const uint32_t* __restrict__ idx, uint32_t* __restrict__ idx_c,
                                                   const int32_t* __restrict__ mm, int32_t* __restrict__ mm_c,
                                                   const uint32_t* __restrict__ orig, uint32_t* __restrict__ orig_c,
                                                   uint32_t T) {
    for (uint32_t i = blockIdx.x * BS + threadIdx.x; i < T; i += gridDim.x * BS) {
        idx_c[3 * (size_t)i] = idx[3 * (size_t)i];
        idx_c[3 * (size_t)i + 1] = idx[3 * (size_t)i + 1];
        idx_c[3 * (size_t)i + 2] = idx[3 * (size_t)i + 2];
        mm_c[i] = mm[i];
        orig_c[i] = orig[i];
    }
}

// rearrange_indices / rearrange_map (src/kernel/bvh-builder.cl:49-72) plus
// the sorted triangle records used by traversal and refit, and the
// original-id map (composition of every build's permutation).
__global__ __launch_bounds__(BS) void k_rearrange(const uint32_t* __restrict__ perm, const uint32_t* __restrict__ idx,
                                                  uint32_t* __restrict__ idx_out, const int32_t* __restrict__ mm,
                                                  int32_t* __restrict__ mm_out, const uint32_t* __restrict__ orig,
                                                  uint32_t* __restrict__ orig_out, const float4* __restrict__ pos,
                                                  float4* __restrict__ tri, uint32_t T) {
    uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i >= T) return;
    uint32_t p = perm[i];
    uint32_t a = idx[3 * (size_t)p], b = idx[3 * (size_t)p + 1], c = idx[3 * (size_t)p + 2];
    idx_out[3 * (size_t)i] = a;
    idx_out[3 * (size_t)i + 1] = b;
    idx_out[3 * (size_t)i + 2] = c;
    mm_out[i] = mm[p];
    orig_out[i] = orig[p];
    float4 pa = pos[a], pb = pos[b], pc = pos[c];
    tri[3 * (size_t)i] = make_float4(pa.x, pa.y, pa.z, __uint_as_float(a));
    tri[3 * (size_t)i + 1] = make_float4(pb.x, pb.y, pb.z, __uint_as_float(b));
    tri[3 * (size_t)i + 2] = make_float4(pc.x, pc.y, pc.z, __uint_as_float(c));
}

// Triangle records from the current index buffer, identity order (the SAH
// build).
__global__ __launch_bounds__(BS) void k_tri_records(const uint32_t* __restrict__ idx, const float4* __restrict__ pos,
                                                    float4* __restrict__ tri, uint32_t T) {
    uint32_t i = blockIdx.x * BS + threadIdx.x;
    if (i >= T) return;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t a = idx[3 * (size_t)i + k];
        float4 p = pos[a];
        tri[3 * (size_t)i + k] = make_float4(p.x, p.y, p.z, __uint_as_float(a));
    }
}

// ------------------------------------------------------------ tree phase --
// The reference splits a range [l, r] of sorted positions whose first and
// last codes differ, and which holds more than min_leaf + 2 triangles, at the
// highest differing bit, after the last position s without that bit
// (find_middle, src/kernel/bvh-builder.cl:484-552), and numbers the children
// level by level in the order of their parents (process_task, :582-671).
// Instead of one launch per level, every inner node is found by its split s,
// which no other node shares:
//   its range is that of the codes that agree with code[s] above the bit in
//     which code[s] and code[s + 1] differ (k_spans);
//   its parent is the split at l - 1 or at r, whichever's codes agree in more
//     bits, and its level the number of its ancestors, from bit masks that a
//     scan carries (k_spans);
//   the nodes of one level lie in the order of their splits, so its rank among
//     all inner nodes in (level, split) order, a stable counting sort by level,
//     gives its children's numbers 1 + 2 rank and 2 + 2 rank (k_ranks), and
//     with its parent's rank its own;
//   the box of a node is the union of the triangle boxes of its range, in
//     any order (k_boxes, k_cross).
// A build was bound by its launches (55, a few microseconds each) and, when
// large, by the chains of dependent reads in each level's tiles; now it has 15
// launches (of 30-bit codes) and no chain longer than one search.  Whole builds,
// back to back, before and now, the wide records included: 65k triangles 259
// and 103 us, 8M triangles 2198 and 1684 us; refit of 1M 145 and 123 us.

// Split s of the nodes: {l, r, flags | level << 2, -}, then (k_boxes) {l, r,
// node, children}.  Flags: bit 0 the left child is a leaf, bit 1 the right.
constexpr uint32_t SPAN_LEFT = 0x40000000u, SPAN_RIGHT = 0x80000000u, SPAN_NUM = 0x3fffffffu;

// Ancestors as masks.  D(k) is the number of leading bits in which code[k] and
// code[k + 1] agree.  Split k is an ancestor of split s iff D(k) is below every
// D from s up to k, and the ancestors of a node have different D, so the
// level is the number of bits of two masks: the D that are new minima walking
// left from s, and walking right, below D(s).  Appending a D to a walk drops the
// mask's bits from D up and sets bit D; such maps compose to maps of the same
// form (min, mask), so one scan per direction gives every split's masks.
struct Walk {
    uint32_t least, mask;  // least D met (32: none), new minima
};
__device__ __forceinline__ uint32_t bits_below(uint32_t n) { return n >= 32u ? 0xffffffffu : (1u << n) - 1u; }
// The walk over `far`, then the nearer `near`.
__device__ __forceinline__ Walk walk_on(Walk far, Walk near) {
    return Walk{far.least < near.least ? far.least : near.least, (far.mask & bits_below(near.least)) | near.mask};
}

// First position of [0, at] with a code >= want, given codes[at] >= want: four
// ways a step, so the chain of dependent reads is log4 of the range.
__device__ __forceinline__ int first_from(const uint32_t* __restrict__ codes, int at, uint32_t want) {
    int lo = -1, hi = at;  // codes[lo] < want <= codes[hi]
    while (hi - lo > 1) {
        const int q = (hi - lo) >> 2, m1 = lo + (q ? q : 1), m2 = lo + ((hi - lo) >> 1), m3 = hi - (q ? q : 1);
        const bool g1 = codes[m1] >= want, g2 = codes[m2] >= want, g3 = codes[m3] >= want;
        const int l = g1 ? lo : (g2 ? m1 : (g3 ? m2 : m3));
        hi = g1 ? m1 : (g2 ? m2 : (g3 ? m3 : hi));
        lo = l;
    }
    return hi;
}
// Last position of [at, T) with a code <= want, given codes[at] <= want.
__device__ __forceinline__ int last_up_to(const uint32_t* __restrict__ codes, int at, int T, uint32_t want) {
    int lo = at, hi = T;  // codes[lo] <= want < codes[hi]
    while (hi - lo > 1) {
        const int q = (hi - lo) >> 2, m1 = lo + (q ? q : 1), m2 = lo + ((hi - lo) >> 1), m3 = hi - (q ? q : 1);
        const bool g1 = codes[m1] > want, g2 = codes[m2] > want, g3 = codes[m3] > want;
        const int l = g1 ? lo : (g2 ? m1 : (g3 ? m2 : m3));
        hi = g1 ? m1 : (g2 ? m2 : (g3 ? m3 : hi));
        lo = l;
    }
    return lo;
}

// Ranges, child kinds, parents and levels; one split per thread.  The codes of
// the tile are in LDS, where a range's ends are found in doubling steps from
// its split.  A range that leaves the tile contains the tile's first or last
// code, so its end there depends only on how many leading bits it shares with
// that code: 33 values per edge, found by 33 lanes side by side, the only
// searches in global memory (their chain of dependent reads bounds small
// builds).  The edge's walk mask has the bits where two neighbouring values
// differ, and the parent is on the side whose walk has the larger D below
// the node's own.
__global__ __launch_bounds__(TREE_TILE) void k_spans(const uint32_t* __restrict__ codes, uint4* __restrict__ span,
                                                     uint32_t* __restrict__ par, uint32_t* __restrict__ level, int T,
                                                     uint32_t min_leaf) {
    constexpr int WAVES = TREE_TILE / RTX_WAVE;
    __shared__ uint32_t s_c[TREE_TILE + 1];
    __shared__ Walk s_w[2][WAVES];
    __shared__ int s_end[2][33];
    __shared__ uint32_t s_edge[2];
    const int tid = (int)threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int base = (int)blockIdx.x * TREE_TILE, s = base + tid;
    const int last = base + TREE_TILE <= T ? base + TREE_TILE - 1 : T - 1;
    s_c[tid] = s < T ? codes[s] : 0u;
    if (tid == 0) s_c[TREE_TILE] = base + TREE_TILE < T ? codes[base + TREE_TILE] : 0u;
    __syncthreads();
    if (w < 2) {
        int end = 0;
        if (lane < 33) {
            const uint32_t rest = lane == 32 ? 0u : 0xffffffffu >> lane;  // the bits not shared
            end = w == 0 ? first_from(codes, base, s_c[0] & ~rest)
                         : last_up_to(codes, last, T, s_c[last - base] | rest);
            s_end[w][lane] = end;
        }
        const int next = __shfl_down(end, 1, RTX_WAVE);
        const uint32_t m = (uint32_t)ballot(lane < 32 && next != end);
        if (lane == 0) s_edge[w] = m;
    }
    const bool pair = s < T - 1;
    const uint32_t c0 = s_c[tid], c1 = pair ? s_c[tid + 1] : c0, x = c0 ^ c1;
    const uint32_t D = x ? (uint32_t)__builtin_clz(x) : 32u;
    // scans: the walk over the wave's splits left of this one (up), right of it
    // (down; the tile's last split counts as beyond the edge)
    Walk up{D, x ? 1u << D : 0u}, down = s < last ? up : Walk{32u, 0u};
    for (int off = 1; off < RTX_WAVE; off <<= 1) {
        const Walk u{(uint32_t)__shfl_up((int)up.least, off, RTX_WAVE), (uint32_t)__shfl_up((int)up.mask, off, RTX_WAVE)};
        const Walk v{(uint32_t)__shfl_down((int)down.least, off, RTX_WAVE),
                     (uint32_t)__shfl_down((int)down.mask, off, RTX_WAVE)};
        if (lane >= off) up = walk_on(u, up);
        if (lane + off < RTX_WAVE) down = walk_on(v, down);
    }
    if (lane == 63) s_w[0][w] = up;
    if (lane == 0) s_w[1][w] = down;
    up = Walk{(uint32_t)__shfl_up((int)up.least, 1, RTX_WAVE), (uint32_t)__shfl_up((int)up.mask, 1, RTX_WAVE)};
    down = Walk{(uint32_t)__shfl_down((int)down.least, 1, RTX_WAVE), (uint32_t)__shfl_down((int)down.mask, 1, RTX_WAVE)};
    if (lane == 0) up = Walk{32u, 0u};
    if (lane == 63) down = Walk{32u, 0u};
    // the range inside the tile
    const uint32_t rest = 0xffffffffu >> (D & 31u), low = c0 & ~rest, high = c0 | rest;
    int l = tid, r = tid + 1;
    if (x) {
        int st = 1;
        while (l - st >= 0 && s_c[l - st] >= low) {
            l -= st;
            st <<= 1;
        }
        for (st >>= 1; st; st >>= 1)
            if (l - st >= 0 && s_c[l - st] >= low) l -= st;
        st = 1;
        const int n = last - base + 1;
        while (r + st < n && s_c[r + st] <= high) {
            r += st;
            st <<= 1;
        }
        for (st >>= 1; st; st >>= 1)
            if (r + st < n && s_c[r + st] <= high) r += st;
    }
    __syncthreads();
    if (s >= T) return;
    uint32_t p = NONE, n = NONE;
    if (x) {
        l = l == 0 ? s_end[0][D] : base + l;
        r = r >= last - base ? s_end[1][D] : base + r;
        // inner: more than min_leaf + 2 triangles (the codes differ by construction)
        if ((uint32_t)(r - l + 1) - 2u > min_leaf) {
            // all codes of a child equal: within the tile its end codes, beyond it
            // the run of the edge's code
            const bool same_l = l >= base ? s_c[l - base] == c0 : (s_c[0] == c0 && s_end[0][32] <= l);
            const bool same_r = r <= last   ? s_c[r - base] == c1
                                : s == last ? codes[r] == c1
                                            : (s_c[last - base] == c1 && s_end[1][32] >= r);
            const bool leaf_l = !((uint32_t)(s - l + 1) - 2u > min_leaf && !same_l);
            const bool leaf_r = !((uint32_t)(r - s) - 2u > min_leaf && !same_r);
            Walk wl{32u, s_edge[0]}, wr{32u, s_edge[1]};
            for (int k = 0; k < w; ++k) wl = walk_on(wl, s_w[0][k]);
            for (int k = WAVES - 1; k > w; --k) wr = walk_on(wr, s_w[1][k]);
            const uint32_t ml = walk_on(wl, up).mask & bits_below(D), mr = walk_on(wr, down).mask & bits_below(D);
            p = (ml | mr) == 0u ? (uint32_t)s : (ml > mr ? (uint32_t)(l - 1) : (uint32_t)r);  // the root: itself
            n = (uint32_t)__builtin_popcount(ml | mr);
            span[s] = make_uint4((uint32_t)l, (uint32_t)r, (leaf_l ? 1u : 0u) | (leaf_r ? 2u : 0u) | (n << 2), 0u);
        }
    }
    par[s] = p;
    level[s] = n;
}

// The rank of every split among those of its level (the level in `rel` is
// replaced by it): in-tile by wave ballots, across tiles by one look-back per
// level, as a radix-sort pass ranks digits.  The last tile writes the level
// table.
template <int RANK_ITEMS>
__global__ __launch_bounds__(BS) void k_ranks(uint32_t* __restrict__ rel, uint32_t* status, uint32_t* ticket,
                                              uint32_t* __restrict__ levels, uint32_t T, uint32_t ntiles) {
    __shared__ uint32_t s_wcnt[BS / RTX_WAVE][64];
    __shared__ uint32_t s_pref[64];
    __shared__ uint32_t s_tile;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (tid == 0) s_tile = atomicAdd(ticket, 1u);
    s_wcnt[w][lane] = 0;
    __syncthreads();
    const uint32_t tile = s_tile, base = tile * (BS * RANK_ITEMS);
    uint32_t d[RANK_ITEMS], r[RANK_ITEMS];
#pragma unroll
    for (int j = 0; j < RANK_ITEMS; ++j) {
        const uint32_t s = base + (w * RANK_ITEMS + j) * RTX_WAVE + lane;
        d[j] = s < T ? rel[s] : NONE;
    }
#pragma unroll
    for (int j = 0; j < RANK_ITEMS; ++j) {
        const bool ok = d[j] != NONE;
        uint64_t peers = ballot(ok);
#pragma unroll
        for (int b = 0; b < 6; ++b) {
            const bool bit = (d[j] >> b) & 1u;
            const uint64_t bal = ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint32_t below = lanes_below(peers);
        const uint32_t basec = ok ? s_wcnt[w][d[j]] : 0u;
        r[j] = basec + below;
        if (ok && below == 0) s_wcnt[w][d[j]] = basec + (uint32_t)__builtin_popcountll(peers);
    }
    __syncthreads();
    if (tid < 64) {
        uint32_t tot = 0;
#pragma unroll
        for (int i = 0; i < BS / RTX_WAVE; ++i) {
            const uint32_t c = s_wcnt[i][tid];
            s_wcnt[i][tid] = tot;
            tot += c;
        }
        const uint32_t prefix = lookback_thread(status + tid, tile, tot, 64u);
        s_pref[tid] = prefix;
        if (tile == ntiles - 1) {
            const uint32_t all = prefix + tot, inc = wave_incl_scan(all, tid);
            if (tid < 63) {
                levels[LV_OFF + tid + 1] = 1u + 2u * (inc - all);
                levels[LV_CNT + tid + 1] = 2u * all;
            } else {
                levels[LV_TOTAL] = 1u + 2u * inc;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RANK_ITEMS; ++j) {
        const uint32_t s = base + (w * RANK_ITEMS + j) * RTX_WAVE + lane;
        if (d[j] != NONE) rel[s] = s_pref[d[j]] + s_wcnt[w][d[j]] + r[j];
    }
}

// Triangles from which the ranks use tiles of 4096 splits instead of 1024: the
// look-back over many tiles then costs more than a tile's longer ranking (8M
// splits 55 against 113 us; at 65k the short tiles take 6.8 us).
constexpr uint32_t RANK_WIDE = 1u << 19;

struct Box {
    v3 lo, hi;
};
// NaN is the identity: min and max drop it.
__device__ __forceinline__ Box no_box() {
    const float n = __builtin_nanf("");
    return Box{mk3(n, n, n), mk3(n, n, n)};
}
__device__ __forceinline__ Box join(const Box& a, const Box& b) { return Box{vmin(a.lo, b.lo), vmax(a.hi, b.hi)}; }
__device__ __forceinline__ void put_node(float4* __restrict__ node, uint32_t n, const Box& b, uint32_t w0,
                                         uint32_t w1) {
    node[2 * (size_t)n] = make_float4(b.lo.x, b.lo.y, b.lo.z, __uint_as_float(w0));
    node[2 * (size_t)n + 1] = make_float4(b.hi.x, b.hi.y, b.hi.z, __uint_as_float(w1));
}

// What k_boxes leaves for the ranges that cross tiles (at most 32 nested
// nodes cross one tile edge): per tile its box, and the boxes of its ends that
// such a range takes from it, by their first or last position.
constexpr uint32_t TILE_ENDS = 32;
struct TreeTiles {
    float4* box;      // 2 per tile: {lo, number of tails}{hi, number of heads}
    float4* tails;    // TILE_ENDS x 2 per tile: {lo, first position}{hi, -}: that position to the tile's end
    float4* heads;    // TILE_ENDS x 2 per tile: the tile's start to that position
    uint4* cross;     // TILE_CROSS per tile: crossing nodes {first, last, node, children or NONE for a leaf}
    uint32_t* ncross;  // per tile
};
// Crossing nodes and leaves whose split is in one tile: at most 32 nested
// nodes and a leaf per tile edge.
constexpr uint32_t TILE_CROSS = 2 * (TILE_ENDS + 1);
constexpr size_t TILE_BYTES = (2 + 4 * TILE_ENDS) * sizeof(float4) + TILE_CROSS * sizeof(uint4) + 4;

struct TreeArgs {
    const uint32_t* __restrict__ idx;
    const float4* __restrict__ pos;
    float4* __restrict__ tri;
    uint4* __restrict__ span;
    const uint32_t* __restrict__ par;
    const uint32_t* __restrict__ rel;
    float4* __restrict__ node;
    uint32_t* __restrict__ parent;
    uint32_t* levels;
    TreeTiles tiles;
    uint32_t T;
};

// Boxes of every node whose range lies in one tile, and what the others take
// from the tile.  Round k has the union of every window of 2^k positions in
// LDS; min and max are idempotent, so the box of a range of 2^k to 2^(k+1) - 1
// positions is the union of its first and its last window, and a node costs
// two windows whatever its size and needs no other node's box.  The ranges are
// listed by their round first, so that a round's are taken by dense lanes.
// Build: also the node numbers from the ranks, and the parent array; REFIT:
// the numbers are kept in the spans, and the triangle records are gathered
// again.  Bound by LDS and barrier latency at few tiles (17 us at 65k), by
// the record, span and node traffic at many (8M: 254 us for 0.9 GB).
constexpr int BOX_THREADS = 512, BOX_ITEMS = TREE_TILE / BOX_THREADS, BOX_ROUNDS = 11;
template <bool REFIT>
__global__ __launch_bounds__(BOX_THREADS) void k_boxes(TreeArgs A) {
    __shared__ float s_m[6][TREE_TILE];
    __shared__ uint4 s_span[TREE_TILE];
    __shared__ uint16_t s_list[2 * TREE_TILE + 2 * TILE_ENDS];
    __shared__ uint32_t s_off[64];
    __shared__ uint32_t s_cnt[BOX_ROUNDS], s_at[BOX_ROUNDS + 1];
    __shared__ uint32_t s_tails, s_heads, s_cross;
    const uint32_t tid = threadIdx.x, base = blockIdx.x * TREE_TILE;
    const uint32_t valid = A.T - base < (uint32_t)TREE_TILE ? A.T - base : (uint32_t)TREE_TILE;
    const uint32_t last = base + valid - 1u;  // the tile's last position
    if (tid == 0) s_tails = s_heads = s_cross = 0;
    if (tid < BOX_ROUNDS) s_cnt[tid] = 0;
    if (!REFIT && tid < 64) s_off[tid] = A.levels[LV_OFF + tid];
    const bool one_leaf = !REFIT && A.levels[LV_TOTAL] == 1u;
    Box m[BOX_ITEMS];
    auto put = [&](uint32_t p, const Box& b) {
        s_m[0][p] = b.lo.x, s_m[1][p] = b.lo.y, s_m[2][p] = b.lo.z;
        s_m[3][p] = b.hi.x, s_m[4][p] = b.hi.y, s_m[5][p] = b.hi.z;
    };
    auto get = [&](uint32_t p) {
        return Box{mk3(s_m[0][p], s_m[1][p], s_m[2][p]), mk3(s_m[3][p], s_m[4][p], s_m[5][p])};
    };
#pragma unroll
    for (int j = 0; j < BOX_ITEMS; ++j) {
        const uint32_t p = j * BOX_THREADS + tid, i = base + p;
        m[j] = no_box();
        if (p < valid) {
            float4 v[3];
            if (REFIT) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const uint32_t a = A.idx[3 * (size_t)i + k];
                    const float4 q = A.pos[a];
                    v[k] = make_float4(q.x, q.y, q.z, __uint_as_float(a));
                    A.tri[3 * (size_t)i + k] = v[k];
                }
            } else {
#pragma unroll
                for (int k = 0; k < 3; ++k) v[k] = A.tri[3 * (size_t)i + k];
            }
            m[j].lo = vmin(vmin(xyz(v[0]), xyz(v[1])), xyz(v[2]));
            m[j].hi = vmax(vmax(xyz(v[0]), xyz(v[1])), xyz(v[2]));
        }
        put(p, m[j]);
    }
    __syncthreads();
    // The ranges that the split at tile position p asks for: 0 its node, 1 and
    // 2 its leaf children, 3 the tile's end after it, 4 the tile's start up to
    // it.  False where there is none.
    auto ask = [&](const uint4& q, uint32_t p, int kind, uint32_t& a, uint32_t& b) -> bool {
        const uint32_t s = base + p;
        if (q.z == NONE) return false;
        if (kind == 0) {
            a = q.x;
            b = q.y;
            return true;
        }
        if (q.w == NONE) return false;  // the root is a leaf
        if (kind == 1) {
            a = q.x;
            b = s;
            return (q.w & SPAN_LEFT) != 0u;
        }
        if (kind == 2) {
            a = s + 1u;
            b = q.y;
            return (q.w & SPAN_RIGHT) != 0u;
        }
        if (kind == 3) {
            a = s + 1u;
            b = last;
            return q.y > last && s < last;
        }
        a = base;
        b = s;
        return q.x < base && s < last;
    };
    uint32_t slot[BOX_ITEMS][5];  // round << 16 | place in the round's list; NONE: not listed
#pragma unroll
    for (int j = 0; j < BOX_ITEMS; ++j) {
        const uint32_t p = j * BOX_THREADS + tid, s = base + p;
        uint4 q = make_uint4(0, 0, NONE, 0);  // {l, r, node, children}; node NONE: no node splits here
        if (s < A.T) {
            if (REFIT) {
                q = A.span[s];
            } else {
                const uint32_t up = A.par[s];
                if (up != NONE) {
                    q = A.span[s];
                    const uint32_t d = q.z >> 2, c = s_off[d + 1u] + 2u * A.rel[s];
                    const uint32_t n = up == s ? 0u : s_off[d] + 2u * A.rel[up] + (s > up ? 1u : 0u);
                    q = make_uint4(q.x, q.y, n, c | ((q.z & 1u) ? SPAN_LEFT : 0u) | ((q.z & 2u) ? SPAN_RIGHT : 0u));
                    A.parent[c] = n;
                    A.parent[c + 1u] = n;
                } else if (one_leaf && s == A.T - 1u) {
                    q = make_uint4(0u, s, 0u, NONE);  // the root is a leaf
                }
                A.span[s] = q;
            }
        }
        s_span[p] = q;
#pragma unroll
        for (int kind = 0; kind < 5; ++kind) {
            uint32_t a, b;
            slot[j][kind] = NONE;
            if (!ask(q, p, kind, a, b)) continue;
            if (kind < 3 && (a < base || b > last)) {
                const uint32_t k = atomicAdd(&s_cross, 1u), c = q.w & SPAN_NUM;
                if (k < TILE_CROSS)
                    A.tiles.cross[(size_t)blockIdx.x * TILE_CROSS + k] =
                        make_uint4(a, b, kind == 0 ? q.z : c + (uint32_t)kind - 1u,
                                   kind == 0 && q.w != NONE ? c : NONE);
            } else {
                const uint32_t k = 31u - (uint32_t)__builtin_clz(b - a + 1u);
                slot[j][kind] = (k << 16) | atomicAdd(&s_cnt[k], 1u);
            }
        }
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t at = 0;
        for (int k = 0; k < BOX_ROUNDS; ++k) {
            s_at[k] = at;
            at += s_cnt[k];
        }
        s_at[BOX_ROUNDS] = at;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < BOX_ITEMS; ++j)
#pragma unroll
        for (int kind = 0; kind < 5; ++kind)
            if (slot[j][kind] != NONE)
                s_list[s_at[slot[j][kind] >> 16] + (slot[j][kind] & 0xffffu)] =
                    (uint16_t)((kind << 10) | (j * BOX_THREADS + tid));
    float4* const tails = A.tiles.tails + (size_t)blockIdx.x * 2 * TILE_ENDS;
    float4* const heads = A.tiles.heads + (size_t)blockIdx.x * 2 * TILE_ENDS;
    __syncthreads();
    for (int k = 0; k < BOX_ROUNDS; ++k) {
        const uint32_t len = 1u << k;
        for (uint32_t i = s_at[k] + tid; i < s_at[k + 1]; i += BOX_THREADS) {
            const uint32_t p = s_list[i] & (TREE_TILE - 1u);
            const int kind = (int)(s_list[i] >> 10);
            const uint4 q = s_span[p];
            uint32_t a = 0, b = 0;
            ask(q, p, kind, a, b);
            const Box box = join(get(a - base), get(b + 1u - len - base));
            const uint32_t c = q.w & SPAN_NUM;
            if (kind == 0) {
                if (q.w == NONE)
                    put_node(A.node, 0u, box, 0u, A.T);
                else
                    put_node(A.node, q.z, box, c, 0u);
            } else if (kind < 3) {
                put_node(A.node, c + (uint32_t)kind - 1u, box, a, b - a + 1u);
            } else if (kind == 3) {
                const uint32_t t = atomicAdd(&s_tails, 1u);
                if (t < TILE_ENDS) put_node(tails, t, box, a, 0u);
            } else {
                const uint32_t t = atomicAdd(&s_heads, 1u);
                if (t < TILE_ENDS) put_node(heads, t, box, b, 0u);
            }
        }
        if (k == BOX_ROUNDS - 1) break;
        // windows of 2^(k+1): mine and the one 2^k further on
#pragma unroll
        for (int j = 0; j < BOX_ITEMS; ++j) {
            const uint32_t p = j * BOX_THREADS + tid + len;
            if (p < (uint32_t)TREE_TILE) m[j] = join(m[j], get(p));
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < BOX_ITEMS; ++j) put(j * BOX_THREADS + tid, m[j]);
        __syncthreads();
    }
    __syncthreads();
    // the last window at position 0 covers the tile
    if (tid == 0) {
        put_node(A.tiles.box, blockIdx.x, m[0], s_tails, s_heads);
        A.tiles.ncross[blockIdx.x] = s_cross;
    }
}

// Boxes of the nodes whose range crosses tiles, one wave each: the tail of
// the first tile, the boxes of the tiles between, the head of the last.
__global__ __launch_bounds__(BS) void k_cross(float4* __restrict__ node, TreeTiles tiles, uint32_t T) {
    const uint32_t lane = threadIdx.x & 63, n = tiles.ncross[blockIdx.x];
    for (uint32_t k = threadIdx.x >> 6; k < n; k += BS / RTX_WAVE) {
        const uint4 q = tiles.cross[(size_t)blockIdx.x * TILE_CROSS + k];
        const uint32_t ta = q.x / TREE_TILE, tb = q.y / TREE_TILE;
        Box b = no_box();
        for (uint32_t t = ta + 1u + lane; t < tb; t += RTX_WAVE)
            b = join(b, Box{xyz(tiles.box[2 * (size_t)t]), xyz(tiles.box[2 * (size_t)t + 1])});
        // lanes 0..31: the entries of the first tile's tails; 32..63: the last tile's heads
        const bool first = lane < TILE_ENDS;
        const uint32_t t = first ? ta : tb, i = lane & (TILE_ENDS - 1u);
        const bool whole = first ? q.x % TREE_TILE == 0u : (q.y + 1u == T || (q.y + 1u) % TREE_TILE == 0u);
        const float4 b0 = tiles.box[2 * (size_t)t], b1 = tiles.box[2 * (size_t)t + 1];
        if (first && ta == tb) {
            // a leaf that starts its tile, listed by the tile before (its parent's
            // split is that tile's last position): a head only
        } else if (whole) {
            b = join(b, Box{xyz(b0), xyz(b1)});
        } else if (i < __float_as_uint(first ? b0.w : b1.w)) {
            const float4* p = (first ? tiles.tails : tiles.heads) + 2 * ((size_t)t * TILE_ENDS + i);
            const float4 p0 = p[0], p1 = p[1];
            if (__float_as_uint(p0.w) == (first ? q.x : q.y)) b = join(b, Box{xyz(p0), xyz(p1)});
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const Box o{mk3(__shfl_xor(b.lo.x, off, RTX_WAVE), __shfl_xor(b.lo.y, off, RTX_WAVE),
                            __shfl_xor(b.lo.z, off, RTX_WAVE)),
                        mk3(__shfl_xor(b.hi.x, off, RTX_WAVE), __shfl_xor(b.hi.y, off, RTX_WAVE),
                            __shfl_xor(b.hi.z, off, RTX_WAVE))};
            b = join(b, o);
        }
        if (lane == 0) put_node(node, q.z, b, q.w == NONE ? q.x : q.w, q.w == NONE ? q.y - q.x + 1u : 0u);
    }
}

// One pass over the child pairs (pair k: nodes 1 + 2k and 2 + 2k), four lanes
// each: the near-child difference right.lo - left.lo of their parent and, where
// the parent is at an even level, its wide record (wide.hpp), number k, one
// slot per lane.  by_level: the tree is level-ordered and its level table gives
// a node's level; else the level is the length of its parent chain.  Reads and
// writes run through the arrays in order (memory bound: 12 to 19 us at 1M
// triangles, by the node count, 163 at 8M).
__global__ __launch_bounds__(BS) void k_pairs(const float4* __restrict__ node, const uint32_t* __restrict__ parent,
                                              float4* __restrict__ delta, float4* __restrict__ wide,
                                              const uint32_t* __restrict__ levels, int by_level) {
    __shared__ uint32_t s_off[64];
    const uint32_t pairs = (levels[LV_TOTAL] - 1u) >> 1, q = threadIdx.x & 3u;
    if (threadIdx.x < 64) s_off[threadIdx.x] = levels[LV_CNT + threadIdx.x] ? levels[LV_OFF + threadIdx.x] : NONE;
    __syncthreads();
    for (uint32_t k = (blockIdx.x * BS + threadIdx.x) >> 2; k < pairs; k += gridDim.x * (BS / 4)) {
        const uint32_t c = 1u + 2u * k + (q >> 1), n = parent[c];
        const float4 f0 = node[2 * (size_t)c], f1 = node[2 * (size_t)c + 1];
        const v3 right = mk3(__shfl_down(f0.x, 2, 4), __shfl_down(f0.y, 2, 4), __shfl_down(f0.z, 2, 4));
        if (q == 0u) {
            const v3 dl = right - xyz(f0);
            delta[n] = make_float4(dl.x, dl.y, dl.z, 0.f);
        }
        if (!wide) continue;
        int d = 0;  // the parent's level
        if (by_level) {
            while (d + 2 < 64 && s_off[d + 2] <= c) ++d;
        } else {
            for (uint32_t p = n; p; p = parent[p]) ++d;
        }
        if (d & 1) continue;
        const uint32_t a = __float_as_uint(f0.w), cnt = __float_as_uint(f1.w);
        float4 g0 = f0, g1 = f1;
        uint32_t ref;
        if (cnt == 0u) {
            const uint32_t g = a + (q & 1u);
            g0 = node[2 * (size_t)g];
            g1 = node[2 * (size_t)g + 1];
            const uint32_t ga = __float_as_uint(g0.w), gc = __float_as_uint(g1.w);
            ref = wide_ref(g, ga, gc);
            // an inner child at level 31 below this slot's node at level 30
            if (d == 28 && gc == 0u &&
                (__float_as_uint(node[2 * (size_t)ga + 1].w) == 0u || __float_as_uint(node[2 * (size_t)ga + 3].w) == 0u))
                ref |= WIDE_DEEP;
        } else if ((q & 1u) == 0u) {
            ref = wide_ref(c, a, cnt);
        } else {
            ref = WIDE_EMPTY;
            g0 = g1 = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
        }
        float4* out = wide + 8 * (size_t)k + 2 * q;
        out[0] = make_float4(g0.x, g0.y, g0.z, __uint_as_float(ref));
        out[1] = make_float4(g1.x, g1.y, g1.z, 0.f);
    }
}

}  // namespace

// ------------------------------------------------------------------ host --
static void write_pairs(rtx_scene* s, hipStream_t st, bool by_level, rtx_ctx* pc) {
    ProfScope ps(pc, st, "lbvh_pairs");
    const uint32_t g = rtx_div_up(2ull * s->T, BS), gmax = (uint32_t)s->ctx->cus * (uint32_t)s->ctx->tune.build_grid;
    hipLaunchKernelGGL(k_pairs, dim3(g > gmax ? gmax : g), dim3(BS), 0, st, s->nodes(), s->b().parent.as<uint32_t>(),
                       s->b().delta.as<float4>(), s->T <= WIDE_MAX_TRIS ? s->b().wide.as<float4>() : nullptr,
                       s->b().levels.as<uint32_t>(), by_level ? 1 : 0);
}

static int32_t lbvh_alloc(rtx_scene* s, uint32_t T, int depth) {
    rtx_ctx* c = s->ctx;
    size_t ncap = 2 * (size_t)T;
    uint32_t passes = (uint32_t)(depth + 7) / 8;
    uint32_t sort_tiles = rtx_div_up(T, SORT_TILE);
    const size_t tree_tiles = rtx_div_up(T, TREE_TILE);
    int32_t e = 0;
    if ((e = s->b().node.reserve(c, ncap * 32 + 64))) return e;
    if ((e = s->b().delta.reserve(c, ncap * 16))) return e;
    if ((e = s->b().parent.reserve(c, ncap * 4))) return e;
    if (T <= WIDE_MAX_TRIS && (e = s->b().wide.reserve(c, (size_t)T * 128))) return e;
    if ((e = s->b().span.reserve(c, (size_t)T * 16))) return e;
    if ((e = s->b().tri.reserve(c, (size_t)T * 48))) return e;
    if ((e = s->b().codes.reserve(c, (size_t)T * 4))) return e;
    if ((e = s->b().perm.reserve(c, (size_t)T * 4))) return e;
    if ((e = s->b().keys_alt.reserve(c, (size_t)T * 4))) return e;
    if ((e = s->b().vals_alt.reserve(c, (size_t)T * 4))) return e;
    if ((e = s->b().centroid.reserve(c, (size_t)T * 16))) return e;
    if ((e = s->b().partials.reserve(c, BOUNDS_GRID * 6 * 4))) return e;
    if ((e = s->b().gbox.reserve(c, 8 * 4))) return e;
    if ((e = s->b().levels.reserve(c, LV_WORDS * 4))) return e;
    if ((e = s->b().tickets.reserve(c, TK_COUNT * 4))) return e;
    if ((e = s->b().sort_hist.reserve(c, 4 * 256 * 4))) return e;
    if ((e = s->b().sort_status.reserve(c, (size_t)passes * sort_tiles * 256 * 4))) return e;
    if ((e = s->b().rank_status.reserve(c, tree_tiles * 64 * 4))) return e;
    if ((e = s->b().tree_tiles.reserve(c, tree_tiles * TILE_BYTES))) return e;
    return 0;
}

// The build's scratch (device memory beyond its inputs and outputs): the
// scene's buffer set holds it for rtx_lbvh_build; the allocation-free build
// carves it from a fixed array instead.
struct BuildScratch {
    uint32_t *keys_alt, *vals_alt;  // radix ping-pong, then the splits' parents and ranks
    float4* centroid;
    float* partials;
    uint32_t *sort_hist, *sort_status, *tickets, *rank_status;
    void* tree_tiles;
};

static BuildScratch scratch_of(BuildSet& b) {
    return BuildScratch{b.keys_alt.as<uint32_t>(),  b.vals_alt.as<uint32_t>(),    b.centroid.as<float4>(),
                        b.partials.as<float>(),     b.sort_hist.as<uint32_t>(),   b.sort_status.as<uint32_t>(),
                        b.tickets.as<uint32_t>(),   b.rank_status.as<uint32_t>(), b.tree_tiles.p};
}

static TreeArgs tree_args(rtx_scene* s, const BuildScratch& W) {
    const size_t tiles = rtx_div_up(s->T, TREE_TILE);
    float4* f = static_cast<float4*>(W.tree_tiles);
    uint4* const cross = reinterpret_cast<uint4*>(f + (2 + 4 * TILE_ENDS) * tiles);
    TreeTiles t{f, f + 2 * tiles, f + (2 + 2 * TILE_ENDS) * tiles, cross,
                reinterpret_cast<uint32_t*>(cross + (size_t)TILE_CROSS * tiles)};
    return TreeArgs{s->idx.as<uint32_t>(), s->pos.as<float4>(),      s->b().tri.as<float4>(),
                    s->b().span.as<uint4>(), W.keys_alt,             W.vals_alt,
                    s->nodes(),            s->b().parent.as<uint32_t>(), s->b().levels.as<uint32_t>(),
                    t,                     s->T};
}

// Boxes of all nodes (REFIT: of the kept topology, from the current
// positions), then the child pairs' differences and wide records.
template <bool REFIT>
static void tree_boxes(rtx_scene* s, hipStream_t st, const BuildScratch& W, rtx_ctx* pc) {
    const TreeArgs A = tree_args(s, W);
    const uint32_t tiles = rtx_div_up(s->T, TREE_TILE);
    {
        ProfScope ps(pc, st, "lbvh_boxes");
        hipLaunchKernelGGL((k_boxes<REFIT>), dim3(tiles), dim3(BOX_THREADS), 0, st, A);
    }
    {
        ProfScope ps(pc, st, "lbvh_cross");
        hipLaunchKernelGGL(k_cross, dim3(tiles), dim3(BS), 0, st, s->nodes(), A.tiles, s->T);
    }
    write_pairs(s, st, true, pc);
}

// Depth and leaf size of a build, clamped as the reference's RendererConfig
// does (src/rt/bvh-builder.cpp:194-199); codes are 32-bit here.
static int32_t build_params(rtx_scene* s, const rtx_lbvh_params* p, int* depth_out, int* min_leaf_out) {
    RTX_REQUIRE(s && s->ctx, RTX_EINVAL, "rtx_lbvh_build: null scene");
    RTX_REQUIRE(s->T > 0 && s->V > 0, RTX_ESTATE, "rtx_lbvh_build: scene has no triangles");
    RTX_REQUIRE(s->T < (1u << 29), RTX_EUNSUPPORTED, "rtx_lbvh_build: more than 2^29 triangles");
    int depth = p ? p->depth : 30;
    int min_leaf = p ? p->min_leaf : 1;
    RTX_REQUIRE(depth <= 32, RTX_EUNSUPPORTED, "rtx_lbvh_build: bvh_depth > 32 needs 64-bit Morton keys");
    *depth_out = depth < 1 ? 1 : depth;
    *min_leaf_out = min_leaf < 1 ? 1 : (min_leaf > 256 ? 256 : min_leaf);
    return RTX_OK;
}

// Sort phase: build state reset, primitive and global bounds, Morton codes,
// radix sort, and the in-place permutation of the scene's index, material
// and id buffers with the triangle records gathered from the positions.  The
// permutation is what chains one build to the next.
// `W` is the scratch; `pc` the context that profiles the launches (null:
// none).  Returns true when the sorted codes and permutation were left in
// W.keys_alt / W.vals_alt (an odd pass count).
static bool build_sort_phase(rtx_scene* s, int depth, hipStream_t st, const BuildScratch& W, rtx_ctx* pc) {
    const uint32_t T = s->T;
    const int rb = (int)s->ctx->tune.sort_bits, items = (int)s->ctx->tune.sort_items;
    const int passes = (depth + rb - 1) / rb;
    const uint32_t sort_tiles = rtx_div_up(T, (uint64_t)BS * items);
    uint32_t* tickets = W.tickets;
    {
        ProfScope ps(pc, st, "lbvh_init");
        const uint32_t nb = (uint32_t)(passes * (size_t)sort_tiles << rb);
        const uint32_t nc = rtx_div_up(T, TREE_TILE) * 64u;
        uint32_t grid = rtx_div_up((uint64_t)(nb > nc ? nb : nc), BS);
        grid = grid < 4 ? 4 : (grid > 2048 ? 2048 : grid);
        hipLaunchKernelGGL(k_build_init, dim3(grid), dim3(BS), 0, st, tickets, (uint32_t)TK_COUNT, W.sort_status, nb,
                           W.rank_status, nc, W.sort_hist, 4u * 256u, s->b().levels.as<uint32_t>(),
                           s->b().parent.as<uint32_t>());
    }
    {
        ProfScope ps(pc, st, "lbvh_prim_bounds");
        uint32_t grid = rtx_div_up(T, BS);
        grid = grid > BOUNDS_GRID ? BOUNDS_GRID : grid;
        hipLaunchKernelGGL(k_prim_bounds, dim3(grid), dim3(BS), 0, st, s->idx.as<uint32_t>(), s->pos.as<float4>(),
                           W.centroid, W.partials, T);
        hipLaunchKernelGGL(k_gbox_reduce, dim3(1), dim3(BS), 0, st, W.partials, grid,
                           s->b().gbox.as<float>());
    }
    {
        ProfScope ps(pc, st, "lbvh_morton");
        uint32_t grid = rtx_div_up(T, BS);
        grid = grid > 1024 ? 1024 : grid;
        hipLaunchKernelGGL(k_morton, dim3(grid), dim3(BS), 0, st, W.centroid, s->b().gbox.as<float>(),
                           s->b().codes.as<uint32_t>(), s->b().perm.as<uint32_t>(), W.sort_hist, T, depth, passes,
                           rb);
    }
    uint32_t *kin = s->b().codes.as<uint32_t>(), *vin = s->b().perm.as<uint32_t>();
    uint32_t *kout = W.keys_alt, *vout = W.vals_alt;
    for (int pass = 0; pass < passes; ++pass) {
        ProfScope ps(pc, st, "lbvh_sort_pass");
        const int shift = rb * pass;
        const int bits = depth - shift < rb ? depth - shift : rb;
        uint32_t* const hist = W.sort_hist + ((size_t)pass << rb);
        uint32_t* const status = W.sort_status + ((size_t)pass * sort_tiles << rb);
#define RTX_SORT_PASS(R, I, N)                                                                                 \
    hipLaunchKernelGGL((k_sort_pass<R, I, N>), dim3(sort_tiles), dim3(N), 0, st, kin, vin, kout, vout, T, shift, \
                       bits, hist, status, tickets + TK_SORT + pass)
        if (rb == 4 && items == 32)
            RTX_SORT_PASS(4, 32, BS);
        else if (rb == 4)
            RTX_SORT_PASS(4, 16, BS);
        else if (items == 32)
            RTX_SORT_PASS(8, 32, BS);
        else if (sort_tiles <= (uint32_t)s->ctx->cus)
            // the tiles fit on the chip side by side (whole builds of 1.05M / 1.5M / 3M
            // triangles: 290 / 391 / 699 us so, 302 / 388 / 689 with small blocks)
            RTX_SORT_PASS(8, 4, 4 * BS);
        else
            RTX_SORT_PASS(8, 16, BS);
#undef RTX_SORT_PASS
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    const bool in_alt = kin != s->b().codes.as<uint32_t>();  // odd pass count
    {
        // permute in place: copy, then gather back into the scene's buffers
        // (no handle swap, so a captured frame chains builds as eager ones do)
        ProfScope ps(pc, st, "lbvh_rearrange");
        uint32_t g = rtx_div_up(T, BS);
        hipLaunchKernelGGL(k_stage_copy, dim3(g > 4096 ? 4096 : g), dim3(BS), 0, st, s->idx.as<uint32_t>(),
                           s->idx_alt.as<uint32_t>(), s->matmap.as<int32_t>(), s->matmap_alt.as<int32_t>(),
                           s->orig.as<uint32_t>(), s->orig_alt.as<uint32_t>(), T);
        hipLaunchKernelGGL(k_rearrange, dim3(rtx_div_up(T, BS)), dim3(BS), 0, st, vin,
                           s->idx_alt.as<uint32_t>(), s->idx.as<uint32_t>(), s->matmap_alt.as<int32_t>(),
                           s->matmap.as<int32_t>(), s->orig_alt.as<uint32_t>(), s->orig.as<uint32_t>(),
                           s->pos.as<float4>(), s->b().tri.as<float4>(), T);
    }
    return in_alt;
}

// Tree phase: ranges, levels and ranks of the splits, then the nodes with
// their boxes.  It reads only the buffer set's own sorted codes and triangle
// records, so it can run beside the next build's sort phase when that one
// writes another set.
static void build_tree_phase(rtx_scene* s, int min_leaf, hipStream_t st, const BuildScratch& W, rtx_ctx* pc) {
    const uint32_t T = s->T, tiles = rtx_div_up(T, TREE_TILE);
    {
        ProfScope ps(pc, st, "lbvh_spans");
        hipLaunchKernelGGL(k_spans, dim3(tiles), dim3(TREE_TILE), 0, st, s->b().codes.as<uint32_t>(),
                           s->b().span.as<uint4>(), W.keys_alt, W.vals_alt, (int)T, (uint32_t)min_leaf);
    }
    {
        ProfScope ps(pc, st, "lbvh_ranks");
        // short tiles while the look-back is short, else fewer of them
#define RTX_RANKS(I)                                                                                                \
    hipLaunchKernelGGL((k_ranks<I>), dim3(rtx_div_up(T, BS * I)), dim3(BS), 0, st, W.vals_alt, W.rank_status,      \
                       W.tickets + TK_RANK, s->b().levels.as<uint32_t>(), T, rtx_div_up(T, BS * I))
        if (T < RANK_WIDE)
            RTX_RANKS(4);
        else
            RTX_RANKS(16);
#undef RTX_RANKS
    }
    tree_boxes<false>(s, st, W, pc);
}

// Sorted codes and permutation left in the scratch's alternates by an odd
// pass count go to the buffer set: by a handle swap when the set owns the
// alternates, by a copy otherwise.
static void settle_sorted(rtx_scene* s, bool in_alt) {
    if (!in_alt) return;
    std::swap(s->b().codes, s->b().keys_alt);
    std::swap(s->b().perm, s->b().vals_alt);
}

int32_t rtx_lbvh_build(rtx_scene* s, const rtx_lbvh_params* p, void* stream) {
    int depth = 30, min_leaf = 1;
    int32_t e = build_params(s, p, &depth, &min_leaf);
    if (e) return e;
    hipStream_t st = s->ctx->pick(stream);
    if ((e = lbvh_alloc(s, s->T, depth))) return e;
    {
        ProfScope whole(s->ctx, st, "LBVH_BUILD");
        settle_sorted(s, build_sort_phase(s, depth, st, scratch_of(s->b()), s->ctx));
        build_tree_phase(s, min_leaf, st, scratch_of(s->b()), s->ctx);
    }
    RTX_CHECK_HIP(hipGetLastError());
    s->built = true;
    s->sah = false;
    s->depth = depth;
    s->min_leaf = min_leaf;
    return RTX_OK;
}

int32_t rtx_lbvh_build_split(rtx_scene* s, const rtx_lbvh_params* p, hipStream_t sort_stream,
                             hipEvent_t sorted, hipStream_t tree_stream) {
    int depth = 30, min_leaf = 1;
    int32_t e = build_params(s, p, &depth, &min_leaf);
    if (e) return e;
    if ((e = lbvh_alloc(s, s->T, depth))) return e;
    settle_sorted(s, build_sort_phase(s, depth, sort_stream, scratch_of(s->b()), s->ctx));
    RTX_CHECK_HIP(hipEventRecord(sorted, sort_stream));
    RTX_CHECK_HIP(hipStreamWaitEvent(tree_stream, sorted, 0));
    build_tree_phase(s, min_leaf, tree_stream, scratch_of(s->b()), s->ctx);
    RTX_CHECK_HIP(hipGetLastError());
    s->built = true;
    s->sah = false;
    s->depth = depth;
    s->min_leaf = min_leaf;
    return RTX_OK;
}

int32_t rtx_lbvh_reserve(rtx_scene* s, int depth) { return lbvh_alloc(s, s->T, depth); }

// ------------------------------------------------ allocation-free build --
// rtx_lbvh_build_noalloc runs the same kernels as rtx_lbvh_build with the
// build scratch carved from `scratch`, a fixed array that every GPU holds for
// the life of the process, so that it calls no allocator.  Sized for
// RTX_LBVH_NOALLOC_MAX_TRIS triangles at any depth <= 32 (4 sort passes of
// 8-bit digits or 8 of 4-bit digits, whose look-back words fit the same space).
// The size is the header's constant, which a program may have compiled in; the
// parts take NA_USED of it.
namespace {
constexpr size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }
constexpr size_t NA_T = RTX_LBVH_NOALLOC_MAX_TRIS;
constexpr size_t NA_SORT_TILES = (NA_T + SORT_TILE - 1) / SORT_TILE;
constexpr size_t NA_TREE_TILES = (NA_T + TREE_TILE - 1) / TREE_TILE;
constexpr size_t NA_USED = 2 * al256(NA_T * 4)                      // keys_alt, vals_alt
                         + al256(NA_T * 16)                         // centroid
                         + al256((size_t)BOUNDS_GRID * 6 * 4)       // partials
                         + al256(4 * 256 * 4)                       // sort_hist
                         + al256(4 * NA_SORT_TILES * 256 * 4)       // sort_status
                         + al256((size_t)TK_COUNT * 4)              // tickets
                         + al256(NA_TREE_TILES * 64 * 4)            // rank_status
                         + al256(NA_TREE_TILES * TILE_BYTES);       // tree_tiles
constexpr size_t NA_BYTES = RTX_LBVH_NOALLOC_SCRATCH_BYTES;
}  // namespace

static_assert(NA_USED <= NA_BYTES, "the scratch holds every part");

static __device__ __align__(256) unsigned char scratch[NA_BYTES];

// Once per context (one device, current when rtx_init calls this): the
// device address of this device's copy of `scratch`.  Host code uses only
// this address, never the array's name.
int32_t rtx_lbvh_scratch_init(rtx_ctx* c) {
    void* ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        rtx_set_error(std::string("rtx_init: hipGetSymbolAddress(build scratch): ") + hipGetErrorString(e));
        return RTX_EDEVICE;
    }
    c->build_scratch = ptr;
    return RTX_OK;
}

static BuildScratch carve_scratch(void* base, uint32_t T) {
    char* p = static_cast<char*>(base);
    auto take = [&](size_t bytes) {
        char* q = p;
        p += al256(bytes);
        return q;
    };
    const size_t sort_tiles = rtx_div_up(T, SORT_TILE), tree_tiles = rtx_div_up(T, TREE_TILE);
    BuildScratch W;
    W.keys_alt = reinterpret_cast<uint32_t*>(take((size_t)T * 4));
    W.vals_alt = reinterpret_cast<uint32_t*>(take((size_t)T * 4));
    W.centroid = reinterpret_cast<float4*>(take((size_t)T * 16));
    W.partials = reinterpret_cast<float*>(take((size_t)BOUNDS_GRID * 6 * 4));
    W.sort_hist = reinterpret_cast<uint32_t*>(take(4 * 256 * 4));
    W.sort_status = reinterpret_cast<uint32_t*>(take(4 * sort_tiles * 256 * 4));
    W.tickets = reinterpret_cast<uint32_t*>(take((size_t)TK_COUNT * 4));
    W.rank_status = reinterpret_cast<uint32_t*>(take(tree_tiles * 64 * 4));
    W.tree_tiles = take(tree_tiles * TILE_BYTES);
    return W;
}

namespace {
__global__ void k_copy_pairs(const uint32_t* __restrict__ ka, const uint32_t* __restrict__ va, uint32_t* __restrict__ kb,
                             uint32_t* __restrict__ vb, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        kb[i] = ka[i];
        vb[i] = va[i];
    }
}
}  // namespace

int32_t rtx_lbvh_build_noalloc(rtx_scene* s, const rtx_lbvh_params* p, void* stream) {
    int depth = 30, min_leaf = 1;
    int32_t e = build_params(s, p, &depth, &min_leaf);
    if (e) return e;
    RTX_REQUIRE(s->T <= RTX_LBVH_NOALLOC_MAX_TRIS, RTX_EINVAL,
                "rtx_lbvh_build_noalloc: more than RTX_LBVH_NOALLOC_MAX_TRIS (1048576) triangles");
    RTX_REQUIRE(s->ctx->build_scratch, RTX_ESTATE, "rtx_lbvh_build_noalloc: context has no build scratch");
    // outputs: the current buffer set, reserved beforehand (rtx_lbvh_build)
    const size_t T = s->T, ncap = 2 * T;
    BuildSet& b = s->b();
    RTX_REQUIRE(b.node.bytes >= ncap * 32 + 64 && b.delta.bytes >= ncap * 16 && b.parent.bytes >= ncap * 4 &&
                    (T > WIDE_MAX_TRIS || b.wide.bytes >= T * 128) &&
                    b.tri.bytes >= T * 48 && b.codes.bytes >= T * 4 && b.perm.bytes >= T * 4 && b.gbox.bytes >= 32 &&
                    b.levels.bytes >= LV_WORDS * 4 && b.span.bytes >= T * 16,
                RTX_ESTATE,
                "rtx_lbvh_build_noalloc: the scene's tree buffers are not reserved for its triangle count "
                "(run rtx_lbvh_build once first)");
    hipStream_t st = s->ctx->pick(stream);
    const BuildScratch W = carve_scratch(s->ctx->build_scratch, s->T);
    if (build_sort_phase(s, depth, st, W, nullptr)) {
        uint32_t g = rtx_div_up(T, BS);
        hipLaunchKernelGGL(k_copy_pairs, dim3(g > 4096 ? 4096 : g), dim3(BS), 0, st, W.keys_alt, W.vals_alt,
                           b.codes.as<uint32_t>(), b.perm.as<uint32_t>(), (uint32_t)T);
    }
    build_tree_phase(s, min_leaf, st, W, nullptr);
    RTX_CHECK_HIP(hipGetLastError());
    s->built = true;
    s->sah = false;
    s->depth = depth;
    s->min_leaf = min_leaf;
    return RTX_OK;
}

// Scene::create_aggregate_bvh with the SAH accelerator (BVH::construct_and_map,
// src/rt/bvh.cpp:126-175): the tree is built on the host from the scene's
// current triangle order, the index buffer, material map and upload ids are
// permuted into its order, and the nodes go to the current buffer set in the
// layout every traversal form reads (children adjacent as the builder
// allocates them, deltas, parents, triangle records).
int32_t rtx_sah_build(rtx_scene* s, void* stream) {
    RTX_REQUIRE(s && s->ctx, RTX_EINVAL, "rtx_sah_build: null scene");
    RTX_REQUIRE(s->T > 0 && s->V > 0, RTX_ESTATE, "rtx_sah_build: scene has no triangles");
    hipStream_t st = s->ctx->pick(stream);
    const uint32_t T = s->T, V = s->V;
    RTX_CHECK_HIP(hipDeviceSynchronize());
    std::vector<float4> p4(V);
    std::vector<uint32_t> idx(3 * (size_t)T), orig(T);
    std::vector<int32_t> mm(T);
    RTX_CHECK_HIP(hipMemcpy(p4.data(), s->pos.p, V * sizeof(float4), hipMemcpyDeviceToHost));
    RTX_CHECK_HIP(hipMemcpy(idx.data(), s->idx.p, idx.size() * 4, hipMemcpyDeviceToHost));
    RTX_CHECK_HIP(hipMemcpy(mm.data(), s->matmap.p, T * 4, hipMemcpyDeviceToHost));
    RTX_CHECK_HIP(hipMemcpy(orig.data(), s->orig.p, T * 4, hipMemcpyDeviceToHost));
    std::vector<float> p3(3 * (size_t)V);
    for (uint32_t v = 0; v < V; ++v) {
        p3[3 * (size_t)v] = p4[v].x;
        p3[3 * (size_t)v + 1] = p4[v].y;
        p3[3 * (size_t)v + 2] = p4[v].z;
    }
    std::vector<rtx_node_ref> nodes;
    std::vector<uint32_t> order;
    uint32_t height = 0;
    int32_t e = rtx_sah_construct(p3.data(), V, idx.data(), T, nodes, order, &height);
    if (e) return e;
    const uint32_t N = (uint32_t)nodes.size();
    std::vector<uint32_t> idx2(idx.size()), orig2(T);
    std::vector<int32_t> mm2(T);
    for (uint32_t i = 0; i < T; ++i) {
        for (int k = 0; k < 3; ++k) idx2[3 * (size_t)i + k] = idx[3 * (size_t)order[i] + k];
        mm2[i] = mm[order[i]];
        orig2[i] = orig[order[i]];
    }
    std::vector<float4> nd(2 * (size_t)N), dl(N, make_float4(0.f, 0.f, 0.f, 0.f));
    std::vector<uint32_t> par(N), lv(LV_WORDS, 0u), depth_of(N, 0u);
    for (uint32_t n = 0; n < N; ++n) {
        const rtx_node_ref& r = nodes[n];
        const bool leaf = r.leaf != 0;
        if (!leaf) RTX_REQUIRE(r.b == r.a + 1, RTX_EUNSUPPORTED, "rtx_sah_build: children not adjacent");
        const uint32_t w0 = r.a, w1 = leaf ? r.b - r.a : 0u;
        float f0, f1;
        std::memcpy(&f0, &w0, 4);
        std::memcpy(&f1, &w1, 4);
        nd[2 * (size_t)n] = make_float4(r.lo[0], r.lo[1], r.lo[2], f0);
        nd[2 * (size_t)n + 1] = make_float4(r.hi[0], r.hi[1], r.hi[2], f1);
        if (!leaf) {
            const rtx_node_ref &L = nodes[r.a], &R = nodes[r.a + 1];
            dl[n] = make_float4(R.lo[0] - L.lo[0], R.lo[1] - L.lo[1], R.lo[2] - L.lo[2], 0.f);
            depth_of[r.a] = depth_of[r.a + 1] = depth_of[n] + 1;  // children follow their parent
        }
        par[n] = r.parent;
        if (depth_of[n] < 64) lv[LV_CNT + depth_of[n]]++;
    }
    lv[LV_TOTAL] = N;
    if ((e = lbvh_alloc(s, T, 30))) return e;
    BuildSet& b = s->b();
    RTX_CHECK_HIP(hipMemcpy(s->idx.p, idx2.data(), idx2.size() * 4, hipMemcpyHostToDevice));
    RTX_CHECK_HIP(hipMemcpy(s->matmap.p, mm2.data(), T * 4, hipMemcpyHostToDevice));
    RTX_CHECK_HIP(hipMemcpy(s->orig.p, orig2.data(), T * 4, hipMemcpyHostToDevice));
    RTX_CHECK_HIP(hipMemcpy(s->nodes(), nd.data(), nd.size() * sizeof(float4), hipMemcpyHostToDevice));
    RTX_CHECK_HIP(hipMemcpy(b.delta.p, dl.data(), dl.size() * sizeof(float4), hipMemcpyHostToDevice));
    RTX_CHECK_HIP(hipMemcpy(b.parent.p, par.data(), N * 4, hipMemcpyHostToDevice));
    RTX_CHECK_HIP(hipMemcpy(b.levels.p, lv.data(), LV_WORDS * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_tri_records, dim3(rtx_div_up(T, BS)), dim3(BS), 0, st, s->idx.as<uint32_t>(),
                       s->pos.as<float4>(), b.tri.as<float4>(), T);
    write_pairs(s, st, false, s->ctx);
    RTX_CHECK_HIP(hipGetLastError());
    RTX_CHECK_HIP(hipStreamSynchronize(st));
    s->built = true;
    s->sah = true;
    // the deepest node's depth: trees of 32 or more levels keep to the
    // traversal forms that follow the MAX_LEVELS rule
    s->depth = (int)std::min<uint32_t>(height, 63);
    return RTX_OK;
}

int32_t rtx_lbvh_refit(rtx_scene* s, void* stream) {
    RTX_REQUIRE(s && s->ctx, RTX_EINVAL, "rtx_lbvh_refit: null scene");
    RTX_REQUIRE(s->built, RTX_ESTATE, "rtx_lbvh_refit: no BVH built");
    RTX_REQUIRE(!s->sah, RTX_ESTATE, "rtx_lbvh_refit: the tree is an SAH tree (refit follows LBVH levels)");
    hipStream_t st = s->ctx->pick(stream);
    // held already unless the tree came from rtx_lbvh_build_noalloc after an
    // rtx_lbvh_build that ran out of memory at its scratch
    int32_t e = s->b().tree_tiles.reserve(s->ctx, rtx_div_up(s->T, TREE_TILE) * TILE_BYTES);
    if (e) return e;
    tree_boxes<true>(s, st, scratch_of(s->b()), s->ctx);
    RTX_CHECK_HIP(hipGetLastError());
    return RTX_OK;
}

int32_t rtx_lbvh_info(rtx_scene* s, uint32_t* node_count, uint32_t* level_counts64) {
    RTX_REQUIRE(s && s->ctx, RTX_EINVAL, "rtx_lbvh_info: null scene");
    RTX_REQUIRE(s->built, RTX_ESTATE, "rtx_lbvh_info: no BVH built");
    uint32_t lv[LV_WORDS];
    RTX_CHECK_HIP(hipStreamSynchronize(s->ctx->stream));
    RTX_CHECK_HIP(hipDeviceSynchronize());
    RTX_CHECK_HIP(hipMemcpy(lv, s->b().levels.p, sizeof lv, hipMemcpyDeviceToHost));
    if (node_count) *node_count = lv[LV_TOTAL];
    if (level_counts64)
        for (int i = 0; i < 64; ++i) level_counts64[i] = (i < 63 && i < s->depth) ? lv[LV_CNT + i + 1] : 0u;
    return RTX_OK;
}

int32_t rtx_read_nodes_ref(rtx_scene* s, rtx_node_ref* out, uint32_t cap, uint32_t* count) {
    uint32_t N = 0;
    int32_t e = rtx_lbvh_info(s, &N, nullptr);
    if (e) return e;
    if (count) *count = N;
    if (!out) return RTX_OK;
    RTX_REQUIRE(cap >= N, RTX_EINVAL, "rtx_read_nodes_ref: capacity below node count");
    std::vector<float4> nd(2 * (size_t)N);
    std::vector<uint32_t> par(N);
    RTX_CHECK_HIP(hipMemcpy(nd.data(), s->nodes(), nd.size() * sizeof(float4), hipMemcpyDeviceToHost));
    RTX_CHECK_HIP(hipMemcpy(par.data(), s->b().parent.p, N * sizeof(uint32_t), hipMemcpyDeviceToHost));
    for (uint32_t n = 0; n < N; ++n) {
        const float4 a = nd[2 * (size_t)n], b = nd[2 * (size_t)n + 1];
        rtx_node_ref& o = out[n];
        o.lo[0] = a.x; o.lo[1] = a.y; o.lo[2] = a.z; o.lo[3] = 0.f;
        o.hi[0] = b.x; o.hi[1] = b.y; o.hi[2] = b.z; o.hi[3] = 0.f;
        uint32_t w0, w1;
        std::memcpy(&w0, &a.w, 4);
        std::memcpy(&w1, &b.w, 4);
        if (w1 == 0) {  // internal
            o.a = w0;
            o.b = w0 + 1;
            o.leaf = 0;
        } else {
            o.a = w0;
            o.b = w0 + w1;
            o.leaf = 1;
        }
        o.parent = n == 0 ? 0u : par[n];
        o.split_axis = 0;
        o.pad[0] = o.pad[1] = 0;
    }
    return RTX_OK;
}
