"""The work that users of this library have it do, as cases to time and compare.

Each case goes through the public binding (tesina-rt_amd/rtx) as a program
does: `prepare` uploads a scene, builds its tree and makes the bundles,
renderers or graphs such a program keeps, `run` is one pass.  The library's
results stay on the device; `run` hands back readers of them (`Outputs`), so
a pass holds no copy to the host that a rendering program would not make,
and whoever looks at an output gets it whole.

Scenes are the generators of rtx.scenes (sphere sets, water surfaces, the
small heightfield-and-sphere scene) and soups of small triangles, at the
sizes that the tests and bench.py use: 10 thousand to 8 million triangles,
256x256 to 1920x1080 pixels, 0 to 4 bounces.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tesina-rt_amd"))
import rtx  # noqa: E402
from rtx import scenes  # noqa: E402

_context = None


def context():
    """One context for the process, as a program has."""
    global _context
    if _context is None:
        torch.cuda.init()
        _context = rtx.Context(0)
    return _context


class Outputs(dict):
    """Outputs by name: each value is read from the device when it is looked at.  Keeps the state they live in."""

    def __init__(self, state, readers):
        dict.__init__(self, readers)
        self.state = state

    def __getitem__(self, name):
        return dict.__getitem__(self, name)()


class State:
    """What a program holds between passes; gives the device memory back with itself."""

    def __init__(self, **held):
        self.__dict__.update(held)
        self.owned = []

    def own(self, *handles):
        self.owned.extend(handles)
        return handles[0]

    def __del__(self):
        context().device_sync()
        for h in reversed(self.owned):
            h.destroy()


# ------------------------------------------------------------------- cases --

def listed():
    return [
        # picking and probes: a few thousand rays of a tool or a simulation into a resident scene
        dict(name="trace 4k rays, 85k tris", kind="trace", scene="small", tris=84800, rays=4096, shadow=False),
        # a renderer of the caller's own: scattered rays (ambient occlusion, diffuse bounces) and their shadow rays
        dict(name="trace 131k scattered, 1M tris", kind="trace", scene="spheres", tris=1000000, rays=131071,
             shadow=True),
        # an animated surface whose topology is kept: vertices moved on the device, boxes refit
        dict(name="refit 1M water", kind="refit", scene="water", tris=1045458),
        # a small dynamic object rebuilt each frame
        dict(name="build 65k tris", kind="build", scene="water", tris=64800),
        # a large captured mesh or point-splat soup indexed from scratch
        dict(name="build 8M tris", kind="build", scene="soup", tris=8000003),
        # the interactive viewer: a frame asked for, waited for and copied to the host for display
        dict(name="frame 512x512 small plain", kind="frame", mode="plain", scene="small", tris=84800, width=512,
             height=512, bounces=1, rebuild=True, accel="lbvh", images=False),
        # a moving scene in a real-time loop: the whole frame, rebuild included, replayed as a graph; odd sizes
        dict(name="frame 1279x719 300k graph", kind="frame", mode="graph", scene="spheres", tris=300000, width=1279,
             height=719, bounces=2, rebuild=True, accel="lbvh", images=False),
        # the headline workload: 1M triangles, 1080p, Whitted depth 3, rebuilt every frame, frames in flight
        dict(name="frame 1080p 1M pipeline", kind="frame", mode="pipeline", scene="spheres", tris=1000000,
             width=1920, height=1080, bounces=3, rebuild=True, accel="lbvh", images=False),
        # the dynamic scene: 1.05M triangles of water displaced and rebuilt inside the captured frame
        dict(name="frame 720p 1M water", kind="frame", mode="graph", scene="water", tris=1045458, width=1280,
             height=720, bounces=2, rebuild=True, accel="lbvh", images=False),
        # a static, textured scene over the SAH tree with a sky
        dict(name="frame 720p 200k sah textured", kind="frame", mode="async", scene="spheres", tris=200000,
             width=1280, height=720, bounces=3, rebuild=False, accel="sah", images=True),
        # a scene of objects moved rigidly every frame, no rebuild
        dict(name="objects 12x100k 720p", kind="objects", tris=100000, meshes=3, count=12, width=1280, height=720,
             bounces=2),
        # a batch of requests over resident scenes (offline batches, the request server's engine)
        dict(name="batch 12 scenes", kind="batch", scenes=6, frames=12, least=10000, most=500000, bounces=3),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "refit", "build", "build", "frame", "frame", "frame", "objects", "batch"])
    scene = rng.choice(["spheres", "water", "soup"])
    if kind == "trace":
        return dict(kind=kind, scene=scene, tris=_log(rng, 10000, 2000000), rays=_log(rng, 1000, 1000000),
                    shadow=rng.random() < 0.5)
    if kind == "refit":
        return dict(kind=kind, scene="water", tris=_log(rng, 10000, 2000000))
    if kind == "build":
        return dict(kind=kind, scene=scene, tris=_log(rng, 10000, 6000000))
    if kind == "objects":
        return dict(kind=kind, tris=_log(rng, 10000, 100000), meshes=rng.randint(1, 4), count=rng.randint(4, 16),
                    width=rng.randint(255, 1024), height=rng.randint(255, 640), bounces=rng.randint(0, 2))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(2, 6), frames=rng.randint(4, 12), least=10000,
                    most=_log(rng, 20000, 500000), bounces=rng.randint(1, 3))
    mode = rng.choice(["plain", "graph", "async", "pipeline"])
    return dict(kind=kind, mode=mode, scene=rng.choice(["spheres", "water"]), tris=_log(rng, 10000, 900000),
                width=rng.randint(255, 1280), height=rng.randint(255, 720), bounces=rng.randint(0, 2),
                rebuild=mode == "pipeline" or rng.random() < 0.6, accel="lbvh", images=rng.random() < 0.3)


# ------------------------------------------------------------------ inputs --

def _data(kind, tris, seed, res=(256, 256)):
    """Scene data of about `tris` triangles (the generators round to whole spheres and grids)."""
    s = scenes.SEED_BASE + 7919 * (int(seed) % 65521) + 11
    if kind == "small":
        return scenes.config_c1(seed=s)
    if kind == "spheres":
        n = max(2, int(round(tris / 5000)))
        return scenes.config_c2(seed=s, n_spheres=n, res=res)
    if kind == "water":
        n = max(8, int(round(math.sqrt(tris / 2.0))) + 1)
        return scenes.config_c3(seed=s, n=n, res=res)
    # soup: triangles of about the mean spacing, in arbitrary order
    g = torch.Generator().manual_seed(s)
    c = torch.rand((tris, 1, 3), generator=g) * 20 - 10
    d = torch.rand((tris, 3, 3), generator=g) - 0.5
    pos = (c + d * (40.0 / tris ** (1 / 3))).reshape(-1, 3).numpy()
    base = scenes.config_c1(seed=s)
    idx = np.arange(3 * tris, dtype=np.uint32).reshape(-1, 3)
    nrm = np.zeros_like(pos)
    nrm[:, 1] = 1.0
    base.camera = dict(pos=(0.0, 0.0, -30.0), look_at=(0.0, 0.0, 0.0), up=(0.0, 1.0, 0.0), fov=np.pi / 4)
    return scenes.SceneData(pos, nrm, np.zeros((3 * tris, 2), np.float32), idx, np.zeros(tris, np.int32),
                            base.materials, base.lights, base.camera, res[0], res[1], 1)


def _upload(state, sd, still=True):
    s = state.own(rtx.Scene(context()))
    if sd.waves is not None:
        if still:
            sd.pos[:, 1] = scenes.displace_host(sd, 0.5)[:, 1]
        scenes.load(s, sd)
        s.set_waves(sd.waves)
    else:
        scenes.load(s, sd)
    return s


def _scattered(sd, n, seed):
    """n rays from points around the scene's box in random directions, and a few thousand per batch that share an
    origin (probes); an odd share misses everything."""
    r = np.random.default_rng(seed)
    lo, hi = sd.pos.min(0).astype(np.float64), sd.pos.max(0).astype(np.float64)
    size = np.maximum(hi - lo, 0.2 * np.max(hi - lo))
    mid = 0.5 * (lo + hi)
    o = mid + (r.random((n, 3)) - 0.5) * 1.2 * size
    aim = mid + (r.random((n, 3)) - 0.5) * size
    o[: n // 4] = mid + 1.1 * size * np.array([0.3, 1.0, -0.9])
    d = aim - o
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-9)
    ori = np.zeros((n, 4), np.float32)
    dr = np.full((n, 4), 1e36, np.float32)
    ori[:, :3], dr[:, :3] = o, d
    return ori, dr


def _images(seed, n, size):
    r = np.random.default_rng(seed)
    return [r.integers(0, 256, (size, size + 2 * k, 4), dtype=np.uint8) for k in range(n)]


def _rigid(seed, count):
    """Transforms of `count` objects on a loose grid, turned about the y axis, and their inverses."""
    r = np.random.default_rng(seed)
    side = int(math.ceil(math.sqrt(count)))
    tr, inv = np.zeros((count, 4, 4)), np.zeros((count, 4, 4))
    for i in range(count):
        a = r.uniform(0, 2 * np.pi)
        m = np.eye(4)
        m[0, 0], m[0, 2], m[2, 0], m[2, 2] = np.cos(a), np.sin(a), -np.sin(a), np.cos(a)
        m[:3, :3] *= r.uniform(0.3, 0.5)
        m[:3, 3] = (9.0 * (i % side - side / 2), r.uniform(-3, 3), 9.0 * (i // side - side / 2))
        tr[i], inv[i] = m, np.linalg.inv(m)
    return tr.astype(np.float32), inv.astype(np.float32)


# ----------------------------------------------------------------- prepare --

def prepare(case, seed):
    return {"trace": _prepare_trace, "refit": _prepare_build, "build": _prepare_build, "frame": _prepare_frame,
            "objects": _prepare_objects, "batch": _prepare_batch}[case["kind"]](case, seed)


def _prepare_trace(case, seed):
    st = State(kind="trace", shadow=case["shadow"], n=case["rays"])
    sd = _data(case["scene"], case["tris"], seed)
    st.scene = _upload(st, sd)
    st.scene.build()
    st.rays = st.own(rtx.Rays(context(), st.n))
    st.hits = st.own(rtx.Hits(context(), st.n))
    ori, dr = _scattered(sd, st.n, seed)
    st.rays.write(ori, dr)
    return st


def _prepare_build(case, seed):
    st = State(kind=case["kind"])
    sd = _data(case["scene"], case["tris"], seed)
    st.scene = _upload(st, sd)
    st.waves, st.t = sd.waves, 0.25 + (seed % 17) * 0.125
    if case["kind"] == "refit":
        st.scene.build()
    return st


def _prepare_frame(case, seed):
    w, h, b = case["width"], case["height"], case["bounces"]
    st = State(kind="frame", mode=case["mode"], rebuild=case["rebuild"])
    sd = _data(case["scene"], case["tris"], seed, (w, h))
    sd.width, sd.height = w, h
    moving = case["scene"] == "water" and case["rebuild"]
    if case["images"]:
        rows = np.frombuffer(sd.materials.tobytes(), np.int32).reshape(-1, 8).copy()
        rows[:, 7] = np.arange(len(rows)) % 4
        sd.materials = np.frombuffer(rows.tobytes(), np.uint8).copy()
    st.scene = _upload(st, sd, still=not moving)
    if case["images"]:
        st.scene.set_textures(_images(seed, 4, 512))
        st.scene.set_cubemap(_images(seed + 1, 6, 256))
    st.cam = scenes.camera_of(sd)
    if case["accel"] == "sah":
        st.scene.build_sah()
    elif not case["rebuild"]:
        st.scene.build()
    if st.mode == "pipeline":
        st.pipe = st.own(rtx.Pipeline(context(), st.scene, w, h, b, depth=3))
        if moving:
            st.pipe.set_animation(True, 0.0, 1.0 / 60)
        return st
    st.renderer = st.own(rtx.Renderer(context(), w, h, b))
    if moving:
        st.renderer.set_animation(True, 0.0, 1.0 / 60)
    if st.mode == "graph":
        st.renderer.frame_async(st.scene, st.cam, st.rebuild)
        context().sync()
        st.renderer.capture(st.scene, st.cam, st.rebuild)
    return st


def _prepare_objects(case, seed):
    st = State(kind="objects", step=0)
    built = []
    for k in range(case["meshes"]):
        s = _upload(st, _data("water" if k % 3 == 1 else "spheres", case["tris"], seed + 31 * k))
        s.build()
        built.append(s)
    poses = [_rigid(1000 * seed + k, case["count"]) for k in range(4)]
    st.poses = poses
    st.objects = st.own(rtx.Instances(context(), [built[i % len(built)] for i in range(case["count"])], *poses[0]))
    r = np.random.default_rng(seed)
    st.objects.set_materials(rtx.make_materials(
        [(*r.uniform(0.2, 1.0, 3), 0.5, (0.0, 0.6, 0.9)[i % 3], (0.0, 0.0, 1.5)[i % 3])
         for i in range(case["count"])]))
    st.objects.set_lights(rtx.make_lights((0.1, 0.1, 0.1), [
        dict(type=rtx.LIGHT_POINT, pos=(30.0, 60.0, -40.0), color=(0.8, 0.8, 0.8)),
        dict(type=rtx.LIGHT_DIR, dir=(0.0, -0.8, 0.6), color=(0.4, 0.4, 0.4))]))
    w, h = case["width"], case["height"]
    st.cam = rtx.camera_set((0.0, 30.0, -55.0), (0.0, 0.0, 0.0), aspect=w / h)
    st.renderer = st.own(rtx.Renderer(context(), w, h, case["bounces"]))
    return st


def _prepare_batch(case, seed):
    st = State(kind="batch", live=[])
    r = np.random.default_rng(seed)
    sds, built = [], []
    sizes = np.exp(np.linspace(math.log(case["least"]), math.log(case["most"]), case["scenes"]))
    for k, tris in enumerate(sizes):
        sd = _data("water" if k % 2 else "spheres", int(tris), seed + 17 * k)
        s = _upload(st, sd)
        s.build()
        sds.append(sd), built.append(s)
    st.jobs = []
    for i in range(case["frames"]):
        k = i % len(built)
        w, h = [(256, 256), (512, 512), (1280, 720)][i % 3]
        cam = scenes.orbit_camera(sds[k], r.normal(size=3), w, h)
        st.jobs.append((built[k], cam, w, h, 1 + i % case["bounces"]))
    st.wave = st.own(rtx.Wavefront(context(), arena_bytes=12 << 30, max_frames=64))
    return st


# --------------------------------------------------------------------- run --

def run(state):
    return {"trace": _run_trace, "refit": _run_refit, "build": _run_build, "frame": _run_frame,
            "objects": _run_objects, "batch": _run_batch}[state.kind](state)


def _once(read):
    """read(), called at the first look."""
    kept = []

    def get(name):
        if not kept:
            kept.append(read())
        return kept[0][name]
    return get


def _run_trace(st):
    rtx.trace(st.scene, st.rays, st.hits, st.n)
    if st.shadow:
        rtx.trace_shadow(st.scene, st.rays, st.hits, st.n)
    get = _once(lambda: st.hits.read(st.n))
    return Outputs(st, {k: (lambda k=k: get(k)) for k in ("flags", "t", "id", "bary", "n4", "p4", "uv2")})


def _tree(scene):
    def read():
        found, (lo, hi) = scene.nodes(), scene.global_bbox()
        nodes = np.zeros(2 * scene.T, found.dtype)  # a tree's node count varies with the vertices
        nodes[:len(found)] = found
        return dict(lo=nodes["lo"][:, :3], hi=nodes["hi"][:, :3], a=nodes["a"].astype(np.int64),
                    b=nodes["b"].astype(np.int64), parent=nodes["parent"].astype(np.int64), leaf=nodes["leaf"] != 0,
                    indices=scene.indices().astype(np.int64), matmap=scene.matmap(),
                    order=scene.orig_ids().astype(np.int64), box=np.stack([lo, hi]))
    return read


TREE = ("lo", "hi", "a", "b", "parent", "leaf", "indices", "matmap", "order", "box")


def _run_build(st):
    st.scene.build()
    get = _once(_tree(st.scene))
    return Outputs(st, {k: (lambda k=k: get(k)) for k in TREE})


def _run_refit(st):
    st.scene.displace_waves(st.waves, st.t)
    st.scene.refit()
    get, verts = _once(_tree(st.scene)), _once(lambda: dict(zip(("pos", "nrm"), st.scene.vertices())))
    readers = {k: (lambda k=k: get(k)) for k in ("lo", "hi", "a", "b")}
    readers.update({k: (lambda k=k: verts(k)) for k in ("pos", "nrm")})
    return Outputs(st, readers)


def _run_frame(st):
    if st.mode == "plain":  # the viewer shows what it gets: the image is copied to the host in the pass
        stats = st.renderer.frame(st.scene, st.cam, st.rebuild)
        image = st.renderer.fb.rgba8()
        rays = np.array([stats.primary_rays, stats.secondary_rays, stats.shadow_rays], np.int64)
        return dict(image=image, rays=rays, accum=st.renderer.fb.accum().astype(np.int64))
    if st.mode == "pipeline":
        f = st.pipe.frame(st.cam, st.rebuild)

        def pixels(which):
            st.pipe.wait(f)
            return getattr(st.pipe.fb(f), which)()
        return Outputs(st, dict(image=lambda: pixels("rgba8"), accum=lambda: pixels("accum").astype(np.int64)))
    if st.mode == "graph":
        st.renderer.replay()
    else:
        st.renderer.frame_async(st.scene, st.cam, st.rebuild)
    fb = st.renderer.fb
    return Outputs(st, dict(image=fb.rgba8, accum=lambda: fb.accum().astype(np.int64)))


def _run_objects(st):
    st.objects.set_transforms(*st.poses[st.step % len(st.poses)])
    st.step += 1
    stats = st.renderer.frame_instances(st.objects, st.cam)
    fb = st.renderer.fb
    return Outputs(st, dict(
        image=fb.rgba8, accum=lambda: fb.accum().astype(np.int64),
        rays=lambda: np.array([stats.primary_rays, stats.secondary_rays, stats.shadow_rays], np.int64)))


def _run_batch(st):
    if st.live:  # the last batch's frames are read by now: their memory goes to the next
        st.wave.sync()
        st.wave.poll()
        for f in st.live:
            st.wave.release(f)
    st.live = [st.wave.add(s, cam, w, h, b, tag=i, ray_capacity=2 * w * h + 2)
               for i, (s, cam, w, h, b) in enumerate(st.jobs)]
    st.wave.run()
    return Outputs(st, {"image%02d" % i: (lambda f=f: st.wave.rgba8(f)) for i, f in enumerate(st.live)})


# -------------------------------------------------- work, tolerance, exact --

def work(case):
    """Bytes: rays and hits, vertices, indices and the tree's nodes, or pixels, each once.  Flops: one walk from the
    root to a leaf per ray that is known beforehand (box tests of both children on each level, one triangle)."""
    k = case["kind"]

    def walk(tris):
        return 2 * 24 * math.log2(max(2, tris)) + 50
    if k == "trace":
        return dict(bytes=case["rays"] * (32 + 60), flops=case["rays"] * walk(case["tris"]) * (2 if case["shadow"] else 1))
    if k == "refit":
        return dict(bytes=case["tris"] * (12 + 0.5 * (12 + 16 + 32) + 1.5 * 32), flops=case["tris"] * 0.5 * 8 * 20)
    if k == "build":
        verts = 3 if case["scene"] == "soup" else 0.5
        return dict(bytes=case["tris"] * (verts * 12 + 2 * 20 + 1.5 * 32 + 48), flops=case["tris"] * 60)
    if k == "batch":
        px = sum([(65536, 262144, 921600)[i % 3] for i in range(case["frames"])])
        return dict(bytes=px * 16, flops=px * walk(case["most"]))
    px = case["width"] * case["height"]
    if k == "objects":
        return dict(bytes=px * 16, flops=px * walk(case["tris"] * case["count"]))
    rebuilt = case["tris"] * (6 + 40 + 48 + 48) if case["rebuild"] else 0
    return dict(bytes=px * 16 + rebuilt, flops=px * walk(case["tris"]) + (case["tris"] * 60 if rebuilt else 0))


def tolerance(case):
    """Trees, images, ray counts and hit ids are whole numbers of a fixed definition.  Distances, points and normals
    of the hits and displaced vertices are short float32 expressions."""
    if case["kind"] in ("trace", "refit"):
        return {"rel": 2e-6}
    return "exact"


def _exact_hits(case, seed):
    """Distances and points of the closest hits by testing every triangle in float64."""
    sd = _data(case["scene"], case["tris"], seed)
    if sd.waves is not None:
        sd.pos[:, 1] = scenes.displace_host(sd, 0.5)[:, 1]
    ori, dr = _scattered(sd, case["rays"], seed)
    p = torch.from_numpy(sd.pos).cuda().double()[torch.from_numpy(sd.idx.astype(np.int64)).cuda()]
    v0, e1, e2 = p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    o, d = torch.from_numpy(ori).cuda().double()[:, :3], torch.from_numpy(dr).cuda().double()[:, :3]
    best = torch.full((len(o),), float("inf"), dtype=torch.float64, device="cuda")
    rows = max(1, (1 << 25) // len(v0))
    n = torch.linalg.cross(e1, e2)
    for i in range(0, len(o), rows):
        oo, dd = o[i:i + rows, None], d[i:i + rows, None]
        det = -(dd * n[None]).sum(-1)
        s = oo - v0[None]
        c = torch.linalg.cross(s, dd.expand_as(s))
        u = (c * e2[None]).sum(-1) / det
        v = -(c * e1[None]).sum(-1) / det
        t = (s * n[None]).sum(-1) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= 0)
        best[i:i + rows] = torch.where(ok, t, torch.full_like(t, float("inf"))).min(1).values
    hit = torch.isfinite(best)
    t = torch.where(hit, best, torch.zeros_like(best))
    pt = torch.zeros((len(o), 4), dtype=torch.float64, device="cuda")
    pt[:, :3] = torch.where(hit[:, None], o + d * t[:, None], torch.zeros_like(o))
    return dict(flags=None, t=t, id=None, bary=None, n4=None, p4=pt, uv2=None)


def exact(case, seed):
    if case["kind"] == "trace" and case["rays"] * case["tris"] < 1e9:
        return _exact_hits(case, seed)
    if case["kind"] == "build":
        sd = _data(case["scene"], case["tris"], seed)
        if sd.waves is not None:
            sd.pos[:, 1] = scenes.displace_host(sd, 0.5)[:, 1]
        out = dict.fromkeys(TREE)
        p = sd.pos.astype(np.float64)
        out["box"] = np.stack([p.min(0), p.max(0)])
        return out
    if case["kind"] == "refit":
        sd = _data(case["scene"], case["tris"], seed)
        t = 0.25 + (seed % 17) * 0.125
        p = sd.pos.astype(np.float64)
        y, gx, gz = (np.zeros(len(p)) for _ in range(3))
        for a, k, dx, dz, om, ph in sd.waves.astype(np.float64):
            at = k * (dx * p[:, 0] + dz * p[:, 2]) - om * t + ph
            y += a * np.sin(at)
            gx += a * k * dx * np.cos(at)
            gz += a * k * dz * np.cos(at)
        p[:, 1] = y
        n = np.stack([-gx, np.ones_like(y), -gz], 1)
        return dict(lo=None, hi=None, a=None, b=None, pos=p, nrm=n / np.linalg.norm(n, axis=1, keepdims=True))
    return None
