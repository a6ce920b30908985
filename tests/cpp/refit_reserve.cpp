// A refit after builds that ran out of device memory.  This program's own
// hipMalloc stands before the HIP runtime's and refuses one chosen request:
// for every allocation of a growing scene's rtx_lbvh_build in turn, the build
// fails there, the scene takes T triangles (the new count, then the old one),
// rtx_lbvh_build_noalloc builds it where it accepts to, and rtx_lbvh_refit
// must leave the boxes that a scene with an undisturbed build has.
//
//   refit_reserve
// Prints "allocations <n> built <m> refit <k>"; exit status 0 when every refit
// was right.
#include <dlfcn.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "rtx.h"

static int g_left = -1;  // requests still granted; -1: all
static int g_seen = 0;

extern "C" int hipMalloc(void** p, size_t bytes) {
    static auto real = reinterpret_cast<int (*)(void**, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
    ++g_seen;
    if (g_left == 0) {
        *p = nullptr;
        return 2;  // hipErrorOutOfMemory
    }
    if (g_left > 0) --g_left;
    return real(p, bytes);
}

struct Mesh {
    std::vector<float> pos, moved;
    std::vector<uint32_t> idx;
    uint32_t V, T;
};

static Mesh mesh(uint32_t T) {
    Mesh m;
    m.T = T;
    m.V = T / 2 + 3;
    uint32_t x = 12345u + T;
    auto next = [&] { return (x = x * 1664525u + 1013904223u) >> 8; };
    for (uint32_t i = 0; i < 3 * m.V; ++i) m.pos.push_back((float)(next() % 20000) * 0.001f - 10.f);
    for (uint32_t i = 0; i < 3 * T; ++i) m.idx.push_back(next() % m.V);
    for (float p : m.pos) m.moved.push_back(p * 0.75f + 0.5f);
    return m;
}

static int load(rtx_scene* s, const Mesh& m) {
    int e = rtx_scene_set_vertices(s, m.pos.data(), nullptr, nullptr, m.V);
    return e ? e : rtx_scene_set_triangles(s, m.idx.data(), nullptr, m.T);
}

static std::vector<rtx_node_ref> refit_nodes(rtx_ctx* c, rtx_scene* s, const Mesh& m) {
    std::vector<rtx_node_ref> n(2 * (size_t)m.T);
    uint32_t count = 0;
    if (rtx_scene_update_positions(s, m.moved.data(), nullptr) || rtx_lbvh_refit(s, nullptr) || rtx_sync(c, nullptr) ||
        rtx_read_nodes_ref(s, n.data(), (uint32_t)n.size(), &count))
        count = 0;
    n.resize(count);
    return n;
}

static bool same(const std::vector<rtx_node_ref>& a, const std::vector<rtx_node_ref>& b) {
    return !a.empty() && a.size() == b.size() && !std::memcmp(a.data(), b.data(), a.size() * sizeof a[0]);
}

int main() {
    rtx_ctx* c = nullptr;
    if (rtx_init(0, &c)) return std::printf("rtx_init: %s\n", rtx_last_error()), 1;
    const Mesh small = mesh(1500), big = mesh(5000);
    const Mesh* const both[2] = {&big, &small};
    std::vector<rtx_node_ref> want[2];
    for (int k = 0; k < 2; ++k) {
        rtx_scene* s = nullptr;
        if (rtx_scene_create(c, &s) || load(s, *both[k]) || rtx_lbvh_build(s, nullptr, nullptr)) return 1;
        want[k] = refit_nodes(c, s, *both[k]);
        rtx_scene_destroy(s);
    }
    int built = 0, right = 0, allocs = 0;
    bool failed = true;
    for (int at = 0; failed; ++at) {
        rtx_scene* s = nullptr;
        if (rtx_scene_create(c, &s) || load(s, small) || rtx_lbvh_build(s, nullptr, nullptr) || load(s, big)) return 1;
        g_left = at;
        g_seen = 0;
        failed = rtx_lbvh_build(s, nullptr, nullptr) == RTX_ENOMEM;
        allocs = g_seen;
        g_left = -1;
        for (int k = 0; failed && k < 2; ++k) {
            if (load(s, *both[k])) return 1;
            std::printf("allocation %d refused, %u triangles\n", at, both[k]->T);
            std::fflush(stdout);
            if (rtx_lbvh_build_noalloc(s, nullptr, nullptr)) continue;  // outputs not reserved
            ++built;
            if (same(refit_nodes(c, s, *both[k]), want[k])) ++right;
        }
        rtx_scene_destroy(s);
    }
    std::printf("allocations %d built %d refit %d\n", allocs, built, right);
    rtx_shutdown(c);
    return built > 0 && right == built ? 0 : 1;
}
