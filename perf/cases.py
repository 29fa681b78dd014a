"""The measured cases: what a renderer has this library do, over the range of sizes in use.

  trace    one ray queue against a resident scene, closest or any hit (imba_intersect /
           imba_occluded), over random triangles or masked, rotated and scaled instances
  batch    many queues over several scenes in one batched traversal (imba_trace_batch_launch)
  bounce   the queue work between two bounces: compact_hits, then sort_by_material of the hits
  build    the photon hash grid over the photons of one iteration (imba_hashgrid_build)
  query    the k nearest photons within the radius of every camera vertex (imba_hashgrid_query)
  pt       one path-traced frame with next-event shadow rays, captured as a graph (PathTracer)
  vcm      one iteration of vertex connection and merging (VcmRenderer)

Scenes are what a program uploads once and keeps, so states of one case share them; rays,
photons, queries, queues and sample seeds come from the state's seed.  Asynchronous calls of all
states go to one stream, as a program's would.  Hits, photon lists and moved records are fixed
bit for bit by the library's contract, so those outputs are compared exactly.
"""
from __future__ import annotations

import ctypes as C
import functools
import math

import numpy as np
import torch

from imbatracer_amd import native as N
from imbatracer_amd import scene as S
from imbatracer_amd import vcm as V
from imbatracer_amd import workloads as W

FAR = 8.0              # ray length: beyond every scene of the trace and batch cases
GEOMETRY_SEED = 0x1234  # scenes do not depend on a state's seed

# Launch configurations programs use: the default, and the quantized 4-wide tree the launch
# autotuner picks for opaque scenes.
CONFIGS = {"default": None, "q4": N.TraceConfig(256, 16, 0, 0, 4, 1, 0)}


def listed():
    return [
        # a preview tile or a probe: the smallest queue, where the launch counts
        dict(name="trace-small", kind="trace", scene="random", tris=4096, rays=4096, source="camera", any_hit=False,
             tree="default"),
        # a full frame's primary rays over a middle-sized mesh, launched as the autotuner advises
        dict(name="trace-primary", kind="trace", scene="random", tris=65536, rays=1 << 20, source="camera",
             any_hit=False, tree="q4"),
        # the same frame's shadow rays towards a point light, default launch
        dict(name="trace-occluded", kind="trace", scene="random", tris=65536, rays=1 << 20, source="shadow",
             any_hit=True, tree="default"),
        # a diffuse bounce: incoherent rays in an odd number, a larger mesh, default launch
        dict(name="trace-diffuse", kind="trace", scene="random", tris=250000, rays=300007, source="hemisphere",
             any_hit=False, tree="default"),
        # foliage-like content: alpha-masked, rotated and scaled instances
        dict(name="trace-masked", kind="trace", scene="masked", tris=20000, rays=200003, source="camera",
             any_hit=False, tree="default"),
        # tiles of many sessions: queues from 1K rays up over scenes of very different size
        dict(name="batch-queues", kind="batch", queues=48, max_rays=150000, tree="q4"),
        # between two bounces of a full frame: path-tracer states, many materials
        dict(name="bounce-queue", kind="bounce", rays=921600, hit_share=0.7, materials=1026, state=40),
        # photons of one full iteration
        dict(name="photon-build", kind="build", photons=4000000, radius=0.006),
        # a full frame's merge queries, the usual list length
        dict(name="photon-query", kind="query", photons=2000000, queries=600001, radius=0.012, k=10),
        # a served request of the smallest resolution over a small scene
        dict(name="pt-small", kind="pt", side=4, level=3, width=128, height=128, spp=1),
        # a frame over millions of triangles
        dict(name="pt-frame", kind="pt", side=16, level=5, width=640, height=480, spp=1),
        # a bidirectional iteration: light paths, grid, connections and merging
        dict(name="vcm-iteration", kind="vcm", side=8, level=4, width=480, height=360, light_paths=172800, k=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "trace", "batch", "bounce", "build", "query", "pt", "vcm"])
    if kind == "trace":
        scene = rng.choice(["random", "random", "random", "masked"])
        source = rng.choice(["camera", "hemisphere", "shadow"])
        return dict(kind=kind, scene=scene,
                    tris=_log_int(rng, 4096, 250000) if scene == "random" else _log_int(rng, 2000, 20000),
                    rays=_log_int(rng, 4096, 1 << 20) if scene == "random" else _log_int(rng, 4096, 200000),
                    source=source, any_hit=source == "shadow" or rng.random() < 0.2,
                    tree=rng.choice(["default", "q4"]) if scene == "random" else "default")
    if kind == "batch":
        return dict(kind=kind, queues=_log_int(rng, 4, 48), max_rays=_log_int(rng, 5000, 150000),
                    tree=rng.choice(["default", "q4"]))
    if kind == "bounce":
        return dict(kind=kind, rays=_log_int(rng, 4096, 921600), hit_share=round(rng.uniform(0.1, 0.95), 3),
                    materials=_log_int(rng, 3, 1026), state=rng.choice([16, 32, 40, 48]))
    if kind == "build":
        return dict(kind=kind, photons=_log_int(rng, 5000, 4000000), radius=round(rng.uniform(0.004, 0.02), 4))
    if kind == "query":
        return dict(kind=kind, photons=_log_int(rng, 5000, 2000000), queries=_log_int(rng, 500, 600000),
                    radius=round(rng.uniform(0.004, 0.012), 4), k=rng.choice([1, 5, 10, 10, 16, 32, 64]))
    side, level = rng.choice([(4, 3), (4, 4), (8, 3), (8, 4)])
    w, h = _log_int(rng, 96, 640), _log_int(rng, 96, 480)
    if kind == "pt":
        return dict(kind=kind, side=side, level=level, width=w, height=h, spp=rng.choice([1, 1, 2]))
    w, h = min(w, 480), min(h, 360)
    return dict(kind=kind, side=side, level=level, width=w, height=h, light_paths=_log_int(rng, 8192, 172800),
                k=rng.choice([5, 10, 16]))


# ---------------------------------------------------------------------------------------------
# Scenes (kept by the program)
class _Geometry:
    """A built and uploaded scene with its triangles in world space (float32, on the GPU)."""

    def __init__(self, build, tri_points):
        self.build = build
        self.scene = S.Scene(build.desc())
        self.tris = torch.from_numpy(np.ascontiguousarray(tri_points, np.float32)).cuda()  # (n, 3, 3)


@functools.lru_cache(maxsize=None)
def _random_geometry(tris: int):
    build, v, i = W.random_tri_scene(tris, seed=GEOMETRY_SEED)
    return _Geometry(build, v[:, :3][i[:, :3].astype(np.int64)])


@functools.lru_cache(maxsize=None)
def _masked_geometry(tris: int):
    """48 instances of a textured random mesh (checkerboard mask) and a sphere, in the unit cube."""
    rng = np.random.default_rng(GEOMETRY_SEED)
    build = S.SceneBuild()
    v0, i0 = S.random_triangles(tris, GEOMETRY_SEED)
    tc = 3.0 * rng.random((len(v0), 2), dtype=np.float32)
    v1, i1 = S.icosphere(4, 0.4, (0.5, 0.5, 0.5), 1)
    meshes = [(build.add_mesh(v0, i0, tc), v0, i0), (build.add_mesh(v1, i1), v1, i1)]
    yy, xx = np.mgrid[0:16, 0:16]
    build.set_mask(0, ((xx + yy) % 2).astype(np.uint8))
    points = []
    for k in range(48):
        mesh, v, i = meshes[0 if k % 4 else 1]
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        m = np.eye(4)
        m[:3, :3] = q * rng.uniform(0.15, 0.35)
        m[:3, 3] = rng.uniform(0.1, 0.9, 3) - m[:3, :3] @ np.full(3, 0.5)
        build.add_instance(mesh, m.astype(np.float32))
        p = v[:, :3][i[:, :3].astype(np.int64)]
        points.append(p @ m[:3, :3].T + m[:3, 3])
    build.run(N.BUILDER_BINNED_SAH, 2)
    return _Geometry(build, np.concatenate(points))


@functools.lru_cache(maxsize=None)
def _sphere_grid(side: int, level: int):
    s = W.SphereGridScene(side=side, level=level, builder=N.BUILDER_BINNED_SAH, threads=8, specular_fraction=0.3)
    return s, S.Scene(s.desc)


def _geometry(case):
    return _random_geometry(case["tris"]) if case["scene"] == "random" else _masked_geometry(case["tris"])


# ---------------------------------------------------------------------------------------------
# Inputs
class _Dev:
    """A torch tensor handed to the library as a device buffer."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.ptr = C.c_void_p(self.t.data_ptr())


@functools.lru_cache(maxsize=None)
def _stream():
    return N.Stream()


class _View:
    """A device pointer of the library as an array for torch.as_tensor, with the object whose
    memory it is."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (int(ptr), False), "version": 3}


def _tensor(owner, ptr, shape, typestr):
    """The library's memory as a tensor; the tensor keeps its owner (outputs may outlive the state)."""
    t = torch.as_tensor(_View(owner, ptr, shape, typestr), device="cuda")
    t.owner = owner
    return t


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _records(org, direction, tmin, tmax):
    n = org.shape[0]
    r = torch.empty(n, 8, device="cuda")
    r[:, 0:3], r[:, 3] = org, tmin
    r[:, 4:7], r[:, 7] = direction, tmax
    return r


def _camera_rays(g, n):
    """Jittered pinhole rays, row by row, of a camera on a ring around the unit cube."""
    u = _uniform(g, 2).tolist()
    a = 2.0 * math.pi * u[0]
    pos = torch.tensor([0.5 + 1.8 * math.sin(a), 0.2 + 0.6 * u[1], 0.5 - 1.8 * math.cos(a)], device="cuda")
    fwd = torch.nn.functional.normalize(torch.tensor([0.5, 0.5, 0.5], device="cuda") - pos, dim=0)
    right = torch.nn.functional.normalize(torch.linalg.cross(fwd, torch.tensor([0.0, 1.0, 0.0], device="cuda")), dim=0)
    up = torch.linalg.cross(right, fwd)
    w = max(1, math.isqrt(n))
    h = -(-n // w)
    at = torch.arange(n, device="cuda")
    jitter = _uniform(g, n, 2)
    half = math.tan(math.radians(25.0))
    x = (((at % w) + jitter[:, 0]) / w * 2.0 - 1.0) * half
    y = (1.0 - ((at // w) + jitter[:, 1]) / h * 2.0) * half
    d = torch.nn.functional.normalize(fwd + x[:, None] * right + y[:, None] * up, dim=1)
    return _records(pos.expand(n, 3), d, 0.0, FAR)


def _hemisphere_rays(g, tris, n):
    """Cosine-weighted rays leaving random points of random triangles on a random side."""
    p = tris[torch.randint(tris.shape[0], (n,), generator=g, device="cuda")]
    s, r = _uniform(g, n).sqrt(), _uniform(g, n)
    org = (1.0 - s)[:, None] * p[:, 0] + (s * (1.0 - r))[:, None] * p[:, 1] + (s * r)[:, None] * p[:, 2]
    nrm = torch.nn.functional.normalize(torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]), dim=1)
    nrm = nrm * torch.where(_uniform(g, n, 1) < 0.5, -1.0, 1.0)
    # a uniform point on the unit sphere added to the normal is cosine distributed around it
    d = nrm + torch.nn.functional.normalize(torch.randn(n, 3, generator=g, device="cuda"), dim=1) * 0.999
    return _records(org, torch.nn.functional.normalize(d, dim=1), 1e-4, FAR)


def _shadow_rays(g, geo, n):
    """From the first hits of camera rays (a point of the cube on a miss) to a point light."""
    rays = _Dev(_camera_rays(g, n))
    hits = _Dev(torch.empty(n, 4, dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    geo.scene.intersect(rays, hits, n)
    t = hits.t.view(torch.float32)[:, 2:3]
    org = torch.where(hits.t[:, :1] >= 0, rays.t[:, 0:3] + t * rays.t[:, 4:7], _uniform(g, n, 3))
    to = torch.tensor([0.5, 2.0, 0.5], device="cuda") + 0.05 * _uniform(g, 1, 3) - org
    dist = to.norm(dim=1)
    return _records(org, to / dist[:, None], 1e-3 * dist, dist * (1.0 - 1e-3))


def _rays(g, geo, source, n):
    if source == "camera":
        return _camera_rays(g, n)
    if source == "hemisphere":
        return _hemisphere_rays(g, geo.tris, n)
    return _shadow_rays(g, geo, n)


def _photon_positions(g, n):
    """Points on the surfaces of 64 spheres of very different size and on a floor, as deposits are."""
    which = torch.randint(0, 80, (n,), generator=g, device="cuda")
    centre = _uniform(g, 80, 3)
    radius = 0.02 + 0.13 * _uniform(g, 80) ** 2
    d = torch.nn.functional.normalize(torch.randn(n, 3, generator=g, device="cuda"), dim=1)
    p = centre[which] + radius[which][:, None] * d
    floor = _uniform(g, n, 3)
    floor[:, 1] = 0.0
    return torch.where((which >= 64)[:, None], floor, p)


class _State:
    pass


def _prepare_trace(case, seed):
    g, s = _generator(seed), _State()
    s.geo, n = _geometry(case), case["rays"]
    s.rays = _Dev(_rays(g, s.geo, case["source"], n))
    s.hits = _Dev(torch.empty(n, 4, dtype=torch.int32, device="cuda"))
    return s


def _hits_out(h):
    f = h.view(torch.float32)
    return {"ids": h[:, 0:2], "t": f[:, 2], "u": f[:, 3]}


def _run_trace(case, s):
    call = s.geo.scene.occluded if case["any_hit"] else s.geo.scene.intersect
    call(s.rays, s.hits, case["rays"], CONFIGS[case["tree"]], _stream())
    return _hits_out(s.hits.t)


BATCH_SCENES = (10000, 30000, 100000, 250000)


def _queue_sizes(case):
    """Log-uniform between 1,000 and max_rays, in an order that mixes small and large queues."""
    n, span = case["queues"], math.log(case["max_rays"] / 1000.0)
    return [int(1000.0 * math.exp(span * ((k * 0.6180339887) % 1.0))) for k in range(n)]


def _prepare_batch(case, seed):
    g, s = _generator(seed), _State()
    sizes = _queue_sizes(case)
    s.rays, items, at = [], [], 0
    s.hits = _Dev(torch.empty(sum(sizes), 4, dtype=torch.int32, device="cuda"))
    for k, n in enumerate(sizes):
        geo = _random_geometry(BATCH_SCENES[k % len(BATCH_SCENES)])
        any_hit = k % 3 == 2
        s.rays.append(_Dev(_rays(g, geo, "shadow" if any_hit else ("camera", "hemisphere")[k % 2], n)))
        items.append((geo.scene, s.rays[-1].ptr, C.c_void_p(s.hits.ptr.value + 16 * at), n, None, any_hit))
        at += n
    torch.cuda.synchronize()
    s.batch = S.TraceBatch(items)
    return s


def _run_batch(case, s):
    s.batch.launch(CONFIGS[case["tree"]], _stream())
    return _hits_out(s.hits.t)


BOUNCE_TRIS = 200000


def _prepare_bounce(case, seed):
    g, s = _generator(seed), _State()
    n, dw = case["rays"], case["state"] // 4
    s.rays = _Dev(_hemisphere_rays(g, _uniform(g, 1000, 3, 3), n))
    hits = torch.randint(0, BOUNCE_TRIS, (n, 4), generator=g, device="cuda", dtype=torch.int32)
    # misses come in runs (the sky) and one by one
    run_miss = (_uniform(g, n // 512 + 1) >= case["hit_share"] ** 0.5).repeat_interleave(512)[:n]
    hits[run_miss | (_uniform(g, n) >= case["hit_share"] ** 0.5), 0] = -1
    s.hits = _Dev(hits)
    s.states = _Dev(torch.randint(0, 1 << 30, (n, dw), generator=g, device="cuda", dtype=torch.int32))
    s.indices = _Dev(torch.randint(0, case["materials"], (BOUNCE_TRIS, 4), generator=g, device="cuda",
                                   dtype=torch.int32))
    s.rays_out, s.hits_out, s.states_out = (_Dev(torch.empty_like(x.t)) for x in (s.rays, s.hits, s.states))
    s.sorted = _Dev(torch.full((n,), -1, dtype=torch.int32, device="cuda"))
    s.starts = _Dev(torch.zeros(case["materials"] + 1, dtype=torch.int32, device="cuda"))
    return s


def _run_bounce(case, s):
    st = _stream()
    n = S.compact_hits(s.rays, s.hits, s.states, case["state"], case["rays"], s.rays_out, s.hits_out, s.states_out, st)
    N.check(N.lib.imba_sort_by_material(s.indices.ptr, BOUNCE_TRIS, s.rays_out.ptr, s.hits_out.ptr, n,
                                        case["materials"], s.sorted.ptr, s.starts.ptr, st.handle), "sort_by_material")
    return {"count": n, "rays": s.rays_out.t.view(torch.int32), "hits": s.hits_out.t, "states": s.states_out.t,
            "sorted": s.sorted.t, "starts": s.starts.t}


def _photon_records(g, n):
    """32-byte photon records (position, path length, direction, pad)."""
    p = torch.zeros(n, 8, device="cuda")
    p[:, 0:3] = _photon_positions(g, n)
    p[:, 4:7] = torch.nn.functional.normalize(torch.randn(n, 3, generator=g, device="cuda"), dim=1)
    return _Dev(p)


def _prepare_build(case, seed):
    g, s = _generator(seed), _State()
    s.photons = _photon_records(g, case["photons"])
    s.grid = S.HashGrid()
    torch.cuda.synchronize()
    s.grid.build(s.photons, 32, 0, case["photons"], case["radius"])
    i = s.grid.info()  # the grid's arrays stay where they are while the photon count does not grow
    s.out = {"ends": _tensor(s.grid, i.cell_ends, (i.table_size,), "<i4"),
             "order": _tensor(s.grid, i.order, (i.photon_count,), "<i4"),
             "positions": _tensor(s.grid, i.positions, (i.photon_count, 4), "<i4")}
    return s


def _prepare_query(case, seed):
    s = _prepare_build(case, seed)
    g = _generator(seed + (1 << 40))
    n, k = case["queries"], case["k"]
    # most queries lie near photons (camera vertices on lit surfaces), neighbours in screen order
    # close to each other; one in sixteen is an empty query slot outside the grid
    base = s.photons.t[torch.randint(case["photons"], (n // 16 + 1,), generator=g, device="cuda"), 0:3]
    q = torch.zeros(n, 16, device="cuda")
    q[:, 0:3] = base.repeat_interleave(16, 0)[:n] + case["radius"] * torch.randn(n, 3, generator=g, device="cuda") * 0.4
    q[_uniform(g, n) < 1.0 / 16.0, 0:3] = math.inf
    s.queries = _Dev(q)
    s.idx = _Dev(torch.full((n, k), -1, dtype=torch.int32, device="cuda"))
    s.dist = _Dev(torch.zeros(n, k, device="cuda"))
    s.count = _Dev(torch.zeros(n, dtype=torch.int32, device="cuda"))
    return s


def _run_build(case, s):
    s.grid.build(s.photons, 32, 0, case["photons"], case["radius"], _stream())
    return s.out


def _run_query(case, s):
    s.grid.query(s.queries, 64, 0, case["queries"], case["k"], s.idx, s.count, s.dist, _stream())
    return {"idx": s.idx.t, "dist": s.dist.t, "count": s.count.t}


def _prepare_pt(case, seed):
    s = _State()
    scene, gpu = _sphere_grid(case["side"], case["level"])
    s.pt = W.PathTracer(scene, case["width"], case["height"], spp=case["spp"], seed_base=seed & 0x7fffffff,
                        trace_cfg=CONFIGS["q4"], gpu_scene=gpu)
    s.pt.build_graph()
    s.image = _tensor(s.pt, s.pt.image.ptr.value, (case["height"], case["width"], 3), "<f4")
    return s


def _run_pt(case, s):
    N.check(N.lib.imba_memset(s.pt.image.ptr, 0, s.pt.image.nbytes, s.pt.stream.handle), "memset")
    counts = s.pt.frame_graph()
    return {"image": s.image, "counts": np.array(counts + [0] * (s.pt.max_path_len - len(counts)), np.int32)}


def _prepare_vcm(case, seed):
    s = _State()
    scene, gpu = _sphere_grid(case["side"], case["level"])
    s.vcm = V.VcmRenderer(scene, case["width"], case["height"], case["light_paths"], k=case["k"],
                          seed_base=seed & 0x7fffffff, light_seed=(seed * 7919 + 1) & 0x7fffffff,
                          trace_cfg=CONFIGS["q4"], shadow_cfg=CONFIGS["q4"], gpu_scene=gpu)
    s.image = _tensor(s.vcm, s.vcm.image.ptr.value, (case["height"], case["width"], 3), "<f4")
    return s


def _run_vcm(case, s):
    s.vcm.clear_image()
    light, camera, vertices = s.vcm.frame()
    return {"image": s.image, "light": np.array(light + [0] * (s.vcm.L - len(light)), np.int32),
            "camera": np.array(camera + [0] * (s.vcm.Lc - len(camera)), np.int32), "vertices": vertices}


_PREPARE = {"trace": _prepare_trace, "batch": _prepare_batch, "bounce": _prepare_bounce, "build": _prepare_build,
            "query": _prepare_query, "pt": _prepare_pt, "vcm": _prepare_vcm}
_RUN = {"trace": _run_trace, "batch": _run_batch, "bounce": _run_bounce, "build": _run_build, "query": _run_query,
        "pt": _run_pt, "vcm": _run_vcm}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    s.case = case
    return s


def run(state):
    return _RUN[state.case["kind"]](state.case, state)


# ---------------------------------------------------------------------------------------------
def _trace_work(rays, tris):
    """Rays in, hits out, every triangle and its share of the tree once; a ray tests two boxes
    (about 12 operations each) per level and a few triangles (about 40 each)."""
    return 48.0 * rays + 80.0 * tris, rays * (24.0 * math.log2(max(tris, 2)) + 120.0)


def work(case):
    kind = case["kind"]
    if kind == "trace":
        b, f = _trace_work(case["rays"], case["tris"] + (20480 if case["scene"] == "masked" else 0))
    elif kind == "batch":
        b, f = _trace_work(sum(_queue_sizes(case)), sum(BATCH_SCENES[:case["queues"]]))
    elif kind == "bounce":
        n = case["rays"]
        b, f = n * (2.0 * (32 + 16 + case["state"]) + case["hit_share"] * (4 + 4 + 4)), 0.0
    elif kind == "build":
        n = case["photons"]
        b, f = n * (12.0 + 4.0 + 16.0 + 2 * 4.0), 20.0 * n
    elif kind == "query":
        nq, k = case["queries"], case["k"]
        # photons within reach: those of a surface patch of the radius
        near = min(case["photons"], case["photons"] * math.pi * case["radius"] ** 2)
        b, f = nq * (12.0 + 8.0 * k + 4.0) + 16.0 * case["photons"], nq * max(near, k) * 8.0
    else:
        pixels = case["width"] * case["height"] * case.get("spp", 1)
        tris = case["side"] ** 2 * 20 * 4 ** case["level"]
        # rays per camera sample (and light path) with the default path lengths
        rays = 7.0 * pixels if kind == "pt" else 6.0 * pixels + 8.0 * case["light_paths"]
        _, f = _trace_work(rays, tris)
        b = 12.0 * case["width"] * case["height"] + 80.0 * tris + 64.0 * rays
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] in ("pt", "vcm"):
        # float32 sums into the image by atomics, whose order is open (seen: 8e-10 and 7e-8), of
        # terms that round to 6e-8 each
        return {"rel": 1e-6, "max": 1e-4}
    return "exact"


# ---------------------------------------------------------------------------------------------
# Reference values in 64 bits
MAX_PAIRS = 2e10


def _exact_closest(tris, rays):
    """Closest hits by testing every triangle (Moeller-Trumbore, edges included), as products of
    the rays' (direction, moment) with per-triangle vectors."""
    p = tris.double()
    v0, e1, e2 = p[:, 0], p[:, 0] - p[:, 1], p[:, 2] - p[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    a_u, a_v, nv = torch.linalg.cross(v0, e2), torch.linalg.cross(v0, e1), (nrm * v0).sum(1)
    t_out, u_out = [], []
    step = max(1, int(2.5e8 // max(1, p.shape[0])))
    for at in range(0, rays.shape[0], step):
        r = rays[at:at + step].double()
        o, d = r[:, 0:3], r[:, 4:7]
        m = torch.linalg.cross(d, o)
        det = d @ nrm.T
        u = (d @ a_u.T - m @ e2.T) / det
        v = (d @ a_v.T - m @ e1.T) / det
        t = (nv[None, :] - o @ nrm.T) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= r[:, 3:4]) & (t <= r[:, 7:8])
        best, arg = torch.where(ok, t, math.inf).min(1)
        hit = torch.isfinite(best)
        t_out.append(torch.where(hit, best, r[:, 7]))
        u_out.append(torch.where(hit, u.gather(1, arg[:, None])[:, 0], 0.0))
    return torch.cat(t_out), torch.cat(u_out)


def _exact_query(case, s):
    """Squared distances of the k nearest photons within the radius, by testing all of them."""
    p, k, r2 = s.photons.t[:, 0:3].double(), case["k"], float(np.float32(case["radius"])) ** 2
    out = torch.zeros(case["queries"], k, dtype=torch.float64, device="cuda")
    kk = min(k, p.shape[0])
    step = max(1, int(2.5e8 // p.shape[0]))
    for at in range(0, case["queries"], step):
        q = s.queries.t[at:at + step, 0:3].double()
        d2 = sum((q[:, a:a + 1] - p[None, :, a]) ** 2 for a in range(3))
        d = torch.topk(d2, kk, dim=1, largest=False).values
        out[at:at + step, :kk] = torch.where(d <= r2, d, 0.0)
    return out


def exact(case, seed):
    if case["kind"] == "trace" and case["scene"] == "random" and not case["any_hit"] \
            and case["rays"] * case["tris"] <= MAX_PAIRS:
        s = prepare(case, seed)
        torch.cuda.synchronize()
        t, u = _exact_closest(s.geo.tris, s.rays.t)
        return {"ids": None, "t": t, "u": u}
    if case["kind"] == "query" and case["photons"] * case["queries"] <= MAX_PAIRS:
        s = prepare(case, seed)
        torch.cuda.synchronize()
        return {"idx": None, "dist": _exact_query(case, s), "count": None}
    # moved records have no rounding; any-hit answers depend on the visiting order; frames are
    # chains of random decisions; larger scenes take too long by testing everything
    return None
