"""The tile edges of the tree phase and the edges of the wide walk's encodings,
against the oracle bit for bit.

Tree phase: tiles of 1024 sorted positions; nodes and runs of equal codes that
cross tile edges, whole trees of one leaf over several tiles, and the triangle
count from which the ranks take wider tiles.

Wide walk: rays with zero and huge direction components whose origins lie on
box planes (an infinite reciprocal is walked node by node, a skipped axis is a
NaN), infinite and tiny tMax, leaves around 15 triangles (the counts a stack
entry holds) and around 32 (from which the whole wave tests a leaf)."""
import numpy as np
import pytest

import oracle as O
from conftest import tuned
from test_gpu_parity import check_build, load_scene, random_scene

pytestmark = pytest.mark.gpu


def _scene(kind, T, seed):
    pos, idx, nrm, uv, mm = random_scene(seed, T)
    if kind == "runs":  # a few triangles, each in a run of up to a thousand equal codes
        rng = np.random.default_rng(seed)
        idx = idx[np.sort(rng.integers(0, max(1, T // 500), T))]
    elif kind == "same":  # one code: a single leaf
        idx = np.repeat(idx[:1], T, axis=0)
    elif kind == "cluster":  # most triangles in one corner: deep and shallow subtrees side by side
        pos[: len(pos) * 3 // 4] *= np.float32(0.001)
    return pos, idx, nrm, uv, mm


@pytest.mark.parametrize("kind,T,depth,min_leaf", [
    ("random", 1023, 30, 1), ("random", 1024, 30, 1), ("random", 1025, 30, 1), ("random", 2049, 32, 3),
    ("random", 5000, 7, 1), ("random", 5000, 1, 1), ("random", 6000, 30, 256), ("runs", 4096, 30, 1),
    ("runs", 5001, 32, 2), ("same", 1024, 30, 1), ("same", 1025, 30, 1), ("same", 3500, 30, 1),
    ("cluster", 9000, 30, 1), ("random", (1 << 19) - 1, 30, 1), ("random", (1 << 19) + 5, 30, 1)])
def test_tree_tiles(ctx, kind, T, depth, min_leaf):
    pos, idx, nrm, uv, mm = _scene(kind, T, 7 + T)
    s = load_scene(ctx, pos, idx, nrm, uv, mm)
    s.build(depth, min_leaf)
    b = O.Build(pos, idx, mm, depth, min_leaf)
    check_build(s, b, T)
    if T < 10000:
        pos2 = (pos * np.float32(0.75) + np.float32(0.5)).astype(np.float32)
        s.update_positions(pos2)
        s.refit()
        b.refit(pos2)
        g = s.nodes()
        assert np.array_equal(g["lo"][:, :3], b.nodes["lo"][:, :3])
        assert np.array_equal(g["hi"][:, :3], b.nodes["hi"][:, :3])
        s.build(depth, min_leaf)  # from the permuted buffers
        b2 = O.Build(pos2, b.idx.reshape(-1, 3), b.matmap, depth, min_leaf)
        g = s.nodes()
        assert np.array_equal(g["a"], b2.nodes["a"]) and np.array_equal(g["lo"][:, :3], b2.nodes["lo"][:, :3])
    s.destroy()


def _odd_rays(rng, pos, n):
    """Axis-parallel and huge directions from vertex coordinates, with all kinds of tMin and tMax."""
    o = pos[rng.integers(0, len(pos), n)].astype(np.float32)
    o += (rng.integers(-1, 2, (n, 3)) * rng.integers(0, 30, (n, 1))).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d[rng.random((n, 3)) < 0.4] = 0.0
    d[rng.random((n, 3)) < 0.05] = -0.0
    d[(d == 0).all(1)] = (0, 0, 1)
    d *= rng.choice(np.array([1.0, 3e6, 1e-5], np.float32), (n, 1), p=[0.8, 0.1, 0.1])
    d[rng.random((n, 3)) < 0.02] = 1e-41  # 1/d overflows
    ori4, dir4 = np.zeros((n, 4), np.float32), np.zeros((n, 4), np.float32)
    ori4[:, :3], dir4[:, :3] = o, d
    ori4[:, 3] = rng.choice(np.array([0.0, 1e-4, 1.0], np.float32), n)
    dir4[:, 3] = rng.choice(np.array([1e36, np.inf, 25.0, 1e-3], np.float32), n)
    return ori4, dir4


def _compare(ctx, s, b, nrm, uv, ori4, dir4, lights):
    import rtx
    n = len(ori4)
    r, h = rtx.Rays(ctx, n), rtx.Hits(ctx, n)
    r.write(ori4, dir4)
    rtx.trace(s, r, h, n)
    rtx.trace_shadow(s, r, h, n)
    g = h.read(n)
    o = O.trace(b, nrm, uv, ori4, dir4)
    o["flags"] = O.trace_shadow(b, O.lights_from(lights), o["flags"], o["p4"])
    for k in ("id", "t", "bary", "flags", "n4", "p4"):
        assert np.array_equal(g[k], o[k], equal_nan=g[k].dtype.kind == "f"), k
    r.destroy()
    h.destroy()
    return o


def _lights():
    import rtx
    return rtx.make_lights((0.1, 0.1, 0.1), [dict(type=rtx.LIGHT_POINT, pos=(2.0, 24.0, -4.0)),
                                             dict(type=rtx.LIGHT_DIR, dir=(0.0, -1.0, 0.0))])


@pytest.mark.parametrize("T,depth,flat,n", [(3000, 30, None, 4097), (3000, 30, 1, 4096), (3000, 32, 0, 1023),
                                            (40000, 30, None, 4096), (2, 30, None, 65)])
def test_wide_walk_odd_rays(ctx, T, depth, flat, n):
    pos, idx, nrm, uv, mm = random_scene(31 + T, T, flat_axis=flat)
    pos = np.round(pos).astype(np.float32) + np.float32(0.0)  # box planes that rays start on
    lights = _lights()
    s = load_scene(ctx, pos, idx, nrm, uv, mm, lights=lights)
    s.build(depth, 1)
    b = O.Build(pos, idx, mm, depth, 1)
    ori4, dir4 = _odd_rays(np.random.default_rng(T + n), pos, n)
    _compare(ctx, s, b, nrm, uv, ori4, dir4, lights)
    s.destroy()


@pytest.mark.parametrize("copies", [3, 4, 5, 14, 15, 16, 17, 31, 32, 33, 70])
def test_wide_walk_leaf_sizes(ctx, copies):
    rng = np.random.default_rng(copies)
    pos, idx, nrm, uv, mm = random_scene(copies, 400)
    idx = np.repeat(idx, copies, axis=0)[rng.permutation(400 * copies)]
    mm = rng.integers(0, 3, len(idx)).astype(np.int32)
    lights = _lights()
    s = load_scene(ctx, pos, idx, nrm, uv, mm, lights=lights)
    s.build()
    b = O.Build(pos, idx, mm, 30, 1)
    o = rng.uniform(-12, 12, (2048, 3))
    d = rng.normal(size=(2048, 3))
    ori4, dir4 = np.zeros((2048, 4), np.float32), np.full((2048, 4), 1e36, np.float32)
    ori4[:, :3], dir4[:, :3] = o, d / np.linalg.norm(d, axis=1, keepdims=True)
    res = _compare(ctx, s, b, nrm, uv, ori4, dir4, lights)
    assert (res["id"] >= 0).sum() > 500
    s.destroy()


def _nested_scene(n=20000, size=0.12):
    """Triangles of one size around centroids that crowd towards a point: a ray through it
    passes most boxes of every level."""
    rng = np.random.default_rng(1)
    c = 0.5 + 0.5 * rng.random((n, 3)) * 2.0 ** -rng.integers(0, 10, (n, 1))
    e = rng.normal(size=(n, 3, 3))
    e = (e - e.mean(1, keepdims=True)) * size
    pos = (c[:, None] + e).reshape(-1, 3).astype(np.float32)
    return pos, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


def _wide_entries(b, o, d):
    """Most stack entries that the ray's wide walk holds before its first leaf (float64 slabs)."""
    lo, hi, leaf = b.nodes["lo"][:, :3].astype(np.float64), b.nodes["hi"][:, :3].astype(np.float64), b.nodes["leaf"]

    def near_first(n):
        a = int(b.nodes["a"][n])
        return (a, a + 1) if np.dot(d, lo[a + 1] - lo[a]) > 0 else (a + 1, a)

    def passes(n):
        t = np.array([(lo[n] - o) / d, (hi[n] - o) / d])
        return max(0.0, t.min(0).max()) <= t.max(0).min()

    stack, most = [0], 1
    while not leaf[stack[-1]]:
        slots = [g for k in near_first(stack.pop()) for g in ((k,) if leaf[k] else near_first(k))]
        stack += [g for g in slots[::-1] if passes(g)]
        most = max(most, len(stack))
    return most


def test_wide_walk_full_stack(ctx):
    """Rays that need more entries than a group's stack holds (32) go on node by node: in the
    scene launches, and in the wavefront frame of the same rays."""
    import rtx
    pos, idx = _nested_scene()
    T = len(idx)
    nrm = np.tile(np.array([[0, 0, -1]], np.float32), (len(pos), 1))
    mm = np.zeros(T, np.int32)
    lights = rtx.make_lights((0.1, 0.1, 0.1), [dict(type=rtx.LIGHT_POINT, pos=(1.5, 1.6, 1.7))])
    s = load_scene(ctx, pos, idx, nrm, None, mm, mats=rtx.make_materials([(0.8, 0.3, 0.2, 0.5, 0.5, 0.0)]),
                   lights=lights)
    s.build(30, 1)
    b = O.Build(pos, idx, mm, 30, 1)
    rng = np.random.default_rng(3)
    d = rng.uniform(0.5, 1.0, (512, 3)).astype(np.float32)
    at = (0.5 + rng.uniform(-0.01, 0.01, (512, 3))).astype(np.float32)
    ori4, dir4 = np.zeros((512, 4), np.float32), np.full((512, 4), 1e36, np.float32)
    ori4[:, :3], dir4[:, :3] = at - d, d
    need = [_wide_entries(b, ori4[i, :3].astype(float), d[i].astype(float)) for i in range(0, 512, 32)]
    assert max(need) > 32, need
    _compare(ctx, s, b, nrm, np.zeros((len(pos), 2), np.float32), ori4, dir4, lights)
    cam = rtx.camera_set((-0.3, -0.35, -0.4), (0.5, 0.5, 0.5), (0, 1, 0), 0.2, 1.0)
    R = rtx.Renderer(ctx, 64, 64, 1)
    st = R.frame(s, cam, rebuild=False)
    wf = rtx.Wavefront(ctx, arena_bytes=1 << 28, max_frames=1)
    fid = wf.add(s, cam, 64, 64, 1)
    wf.run()
    assert np.array_equal(wf.accum(fid), R.fb.accum()) and wf.stats(fid).shadow_rays == st.shadow_rays
    wf.destroy()
    R.destroy()
    s.destroy()


def test_instances_left_to_the_exact_walk(ctx):
    """Rays that leave the wide walk of an instance (a full stack, an infinite reciprocal with an
    infinite tMax) and leaves of all sizes, over sets of one and two chunks of roots: the oracle's
    records, and so those of the loops that walk a ray per lane over the same roots."""
    import rtx
    pos, idx = _nested_scene()
    meshes = [(pos, np.tile(np.float32([0, 0, 1]), (len(pos), 1)), np.zeros((len(pos), 2), np.float32), idx)]
    pos, idx, nrm, uv, _ = random_scene(5, 300)
    pos = np.round(pos).astype(np.float32) + np.float32(0.0)
    meshes.append((pos, nrm, uv, np.repeat(idx, np.arange(300) % 40 + 1, axis=0)))
    scs = [load_scene(ctx, p, i, n, t, np.zeros(len(i), np.int32)) for p, n, t, i in meshes]
    for s in scs:
        s.build(30, 1)
    builds = [O.Build(p, i, None, 30, 1) for p, _, _, i in meshes]
    rng = np.random.default_rng(4)
    ori4, dir4 = _odd_rays(rng, pos, 2048)
    d = rng.uniform(0.5, 1.0, (512, 3)).astype(np.float32)
    ori4[::4, :3], dir4[::4, :3] = 0.5 + rng.uniform(-0.01, 0.01, (512, 3)) - d, d
    ori4[::4, 3], dir4[::4, 3] = 0.0, 1e36
    r, h = rtx.Rays(ctx, 2048), rtx.Hits(ctx, 2048)
    r.write(ori4, dir4)
    for n in (3, 70):
        tr = np.tile(np.eye(4, dtype=np.float32), (n, 1, 1))
        tr[1:, :3, 3] = rng.integers(-20, 20, (n - 1, 3))
        tr[2::3, :3, :3] *= 2.0
        inv = np.linalg.inv(tr).astype(np.float32)
        inst = rtx.Instances(ctx, [scs[i % 2] for i in range(n)], tr, inv)
        inst.set_lights(_lights())
        ms = O.MultiScene(builds, [m[1] for m in meshes], [m[2] for m in meshes],
                          [(i % 2, tr[i], inv[i]) for i in range(n)])
        want = O.trace_multi(ms, ori4, dir4)
        want["flags"] = O.trace_shadow_multi(ms, O.lights_from(_lights()), want["flags"], want["p4"])
        assert (want["id"] >= 0).sum() > 300
        for form, wide in ((0, 1), (1, 1), (1, 0)):
            with tuned(ctx, trace_variant=form, wide_walk=wide):
                inst.trace(r, h, 2048)
                inst.trace_shadow(r, h, 2048)
                got = h.read(2048)
            for k in ("flags", "t", "id", "bary", "n4", "p4", "uv2"):
                assert np.array_equal(got[k], want[k], equal_nan=got[k].dtype.kind == "f"), (n, form, wide, k)
        inst.destroy()
    for x in (r, h, *scs):
        x.destroy()


@pytest.mark.parametrize("T", [1, 4095, 4096, 4097, 70001, 1 << 20, (1 << 20) + 1])
def test_sort_tiles(ctx, T):
    """Edges of the sort's tiles (4096 pairs) and of the count (a tile per CU) up to which a tile
    takes 1024 threads: a stable order, the same as over tiles of 8192."""
    rng = np.random.default_rng(T)
    pos = rng.uniform(-5, 5, (max(3, T // 3), 3)).astype(np.float32)
    idx = rng.integers(0, len(pos), (T, 3)).astype(np.uint32)
    got = []
    for items in (32, 16):
        with tuned(ctx, sort_items=items):
            s = load_scene(ctx, pos, idx, None, None, np.zeros(T, np.int32))
            s.build()
            got.append((s.codes(), s.perm()))
            s.destroy()
    codes, perm = got[1]
    unsorted = np.empty_like(codes)
    unsorted[perm] = codes
    assert np.array_equal(np.argsort(unsorted, kind="stable"), perm)
    assert np.array_equal(got[0][0], codes) and np.array_equal(got[0][1], perm)


def test_frames_without_the_wide_walk(ctx):
    """Every way of rendering the same frames with one lane per ray (wide_walk 0, as over trees without
    wide records) gives the images of the four-lane walk."""
    import rtx
    from rtx import scenes
    sd = scenes.config_c1()
    s = scenes.load(rtx.Scene(ctx), sd)
    w, h = 160, 120
    cam = rtx.camera_set(sd.camera["pos"], sd.camera["look_at"], sd.camera["up"], sd.camera["fov"], w / h)

    def frames():
        out = {}
        R = rtx.Renderer(ctx, w, h, 3)
        for mode in ("plain", "async", "pipelined", "graph"):
            R.set_pipelined(mode == "pipelined")
            if mode == "plain":
                R.frame(s, cam)
            elif mode == "graph":
                R.capture(s, cam)
                for _ in range(2):
                    R.replay()
            else:
                for _ in range(2):
                    R.frame_async(s, cam)
            ctx.sync()
            out[mode] = R.fb.accum()
        R.destroy()
        pl = rtx.Pipeline(ctx, s, w, h, 3, depth=2)
        for _ in range(3):
            last = pl.frame(cam)
        pl.wait(last)
        out["pipeline"] = pl.fb(last).accum()
        pl.destroy()
        return out

    want = frames()
    assert (want["plain"] > 0).any(1).mean() > 0.2
    with tuned(ctx, wide_walk=0):
        got = frames()
    for mode in want:
        assert np.array_equal(got[mode], want[mode]), mode
        assert np.array_equal(got[mode], want["plain"]), mode
    s.destroy()


def test_tree_without_wide_records(ctx):
    """A scene that had wide records, then a mesh of more than 2^25 triangles, which gets none (the
    earlier tree's are still in the buffer): scene, accelerator-copy, wavefront and instance launches
    of the default form give the records of form 0, before and after a refit, and rays straight down
    end on the surface."""
    import rtx
    n, m = 4098, 4098  # 2 * 4097 * 4097 triangles
    x = np.arange(n, dtype=np.float32)

    def mesh(phase):
        y = np.round(8 * np.sin(0.01 * x[:, None] + phase) * np.cos(0.013 * x[None, :])).astype(np.float32)
        pos = np.empty((n, m, 3), np.float32)
        pos[..., 0], pos[..., 1], pos[..., 2] = x[:, None], y, x[None, :]
        return pos.reshape(-1, 3)

    pos = mesh(0.0)
    v = np.arange(n * m, dtype=np.uint32).reshape(n, m)[:-1, :-1].ravel()
    idx = np.empty((2 * len(v), 3), np.uint32)
    for k, o in enumerate((0, m, m + 1)):
        np.add(v, np.uint32(o), out=idx[0::2, k])
    for k, o in enumerate((0, m + 1, 1)):
        np.add(v, np.uint32(o), out=idx[1::2, k])
    T = len(idx)
    assert T > 1 << 25
    mats = rtx.make_materials([(0.8, 0.3, 0.2, 0.5, 0.5, 0.0)])
    lights = rtx.make_lights((0.1, 0.1, 0.1), [dict(type=rtx.LIGHT_POINT, pos=(2000.0, 300.0, 2000.0))])
    p, i, nr, _, _ = random_scene(3, 5000)
    s = load_scene(ctx, p, i, nr, mats=mats, lights=lights)
    s.build()
    # with normals: bounce rays of zero normals are NaN, which pass every box of the tree
    s.set_geometry(pos, idx, np.tile(np.float32([0, 1, 0]), (len(pos), 1)))
    s.build()
    small = load_scene(ctx, p, i, nr, lights=lights)
    small.build()
    rng = np.random.default_rng(8)
    count = 8192
    ori4, dir4 = np.zeros((count, 4), np.float32), np.full((count, 4), 1e36, np.float32)
    ori4[:, 0], ori4[:, 2] = rng.uniform(0, n - 1, (2, count))
    ori4[:, 1] = 50
    dir4[:, :3] = rng.normal(size=(count, 3))
    dir4[:, 1] = -np.abs(dir4[:, 1]) * 0.2
    dir4[: count // 2, :3] = (0, -1, 0)
    r, h = rtx.Rays(ctx, count), rtx.Hits(ctx, count)
    r.write(ori4, dir4)
    inst = rtx.Instances(ctx, [s, small], np.tile(np.eye(4, dtype=np.float32), (2, 1, 1)),
                         np.tile(np.eye(4, dtype=np.float32), (2, 1, 1)))
    inst.set_lights(lights)
    cam = rtx.camera_set((100.0, 60.0, -50.0), (800.0, 0.0, 800.0), (0, 1, 0), np.pi / 4, 1.0)
    bvh = rtx.BVHCopy(ctx)

    def records(trace, shadow):
        trace()
        shadow()
        return h.read(count)

    def everything():
        out = {"scene": records(lambda: rtx.trace(s, r, h, count), lambda: rtx.trace_shadow(s, r, h, count)),
               "copy": records(lambda: rtx.trace(s, r, h, count, bvh=bvh),
                               lambda: rtx.trace_shadow(s, r, h, count, bvh=bvh)),
               "instances": records(lambda: inst.trace(r, h, count), lambda: inst.trace_shadow(r, h, count))}
        wf = rtx.Wavefront(ctx, arena_bytes=1 << 28, max_frames=1)
        fid = wf.add(s, cam, 128, 128, 1)
        wf.run()
        out["wavefront"] = {"accum": wf.accum(fid)}
        wf.destroy()
        return out

    for phase in (0.0, 0.7):
        if phase:
            pos = mesh(phase)
            s.update_positions(pos)
            s.refit()
        bvh.copy(s)
        got = everything()
        with tuned(ctx, trace_variant=0):
            want = everything()
        for what in want:
            for k in want[what]:
                assert np.array_equal(got[what][k], want[what][k], equal_nan=True), (phase, what, k)
        assert np.array_equal(got["copy"]["id"], got["scene"]["id"])
        assert got["wavefront"]["accum"].any()
        down = got["scene"]["t"][: count // 2]
        c = ori4[: count // 2].astype(np.float64)
        ix, iz = np.floor(c[:, 0]).astype(int), np.floor(c[:, 2]).astype(int)
        fx, fz = c[:, 0] - ix, c[:, 2] - iz
        y = pos.reshape(n, m, 3)[..., 1].astype(np.float64)
        y00, y10, y01, y11 = y[ix, iz], y[ix + 1, iz], y[ix, iz + 1], y[ix + 1, iz + 1]
        at = np.where(fx >= fz, y00 + fx * (y10 - y00) + fz * (y11 - y10), y00 + fz * (y01 - y00) + fx * (y11 - y01))
        # t is near 50; its rounding, and that of the vertex differences, are a few units of 4e-6
        assert np.abs(50 - down - at).max() < 1e-3
    for z in (inst, bvh, r, h, s, small):
        z.destroy()
