"""Small queues over the quantized tree are traced with four lanes per ray, and waves of larger ones
go over to that when 16 rays are left: hits equal those of the persistent kernel (one lane per
ray throughout) bit for bit, closest and any hit, and the oracle's closest hits, at the edges of
quads, waves and the largest queue that starts this way, over leaves longer than a quad, stacks
deeper than the LDS part, instances and masks, for device-side counts and batches.  The scenes'
triangles are in general position (or coincide, which no tree tells apart), so the default launch's
closest hits, the BVH2's, are the same.
"""
import numpy as np
import pytest

import oracle
from imbatracer_amd import native as N
from imbatracer_amd import scene as S
from tests import scenes as T

pytestmark = pytest.mark.gpu

Q4 = N.TraceConfig(256, 16, 0, 0, 4, 1, 0)
STRIDED = N.TraceConfig(256, 8, 0, 1, 4, 1, 0)  # one block per CU, rays strided, 8 stack entries in LDS
ONE_LANE = N.TraceConfig(256, 16, 1, 0, 4, 1, 0)  # the persistent kernel
BVH2 = N.TraceConfig(256, 16, 0, 0, 2, 0, 0)
LARGEST = 81920  # on 256 CUs


def _same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.int32), np.ascontiguousarray(b).view(np.int32))


def _stacked():
    """Leaves of up to 13 coincident triangles (equal distances: the smallest id wins)."""
    v, i = S.random_triangles(300, 31)
    tri = v.reshape(-1, 3, 4)
    rng = np.random.default_rng(7)
    tri = np.concatenate([np.repeat(tri[k:k + 1], rng.integers(1, 14), 0) for k in range(len(tri))])
    b = S.SceneBuild()
    b.add_mesh(tri.reshape(-1, 4), np.arange(3 * len(tri), dtype=np.uint32).reshape(-1, 3))
    b.run(N.BUILDER_BINNED_SAH, 1)
    return b


SCENES = {"random": lambda: T.random_tri_scene(20000, N.BUILDER_SBVH)[0], "instanced": T.instanced_scene,
          "masked": T.masked_scene, "stacked": _stacked}


@pytest.mark.parametrize("name", sorted(SCENES))
def test_sizes(gpu, name):
    b = SCENES[name]()
    sc = S.Scene(b.desc())
    box = (-2.0, 2.0) if name == "instanced" else (-0.2, 1.2)
    rays = T.random_rays(LARGEST + 1, seed=8, box=box)
    want, _ = oracle.trace(b.arrays(), rays, threads=8)
    want_any = sc.trace_host(rays, any_hit=True, cfg=ONE_LANE)
    assert (want["tri_id"] >= 0).sum() > 100
    for n in (1, 3, 15, 16, 17, 63, 64, 65, 1000, LARGEST, LARGEST + 1):
        assert _same(sc.trace_host(rays[:n], cfg=Q4), want[:n]), n
        assert _same(sc.trace_host(rays[:n]), want[:n]), n
        assert _same(sc.trace_host(rays[:n], any_hit=True, cfg=Q4), want_any[:n]), n
        assert _same(sc.trace_host(rays[:n], cfg=STRIDED), want[:n]), n
        assert _same(sc.trace_host(rays[:n], any_hit=True, cfg=STRIDED), want_any[:n]), n
    assert _same(sc.trace_host(rays, cfg=BVH2), want)
    assert sc.error_count() == 0


def test_device_counts_and_batches(gpu):
    b = T.instanced_scene()
    sc = S.Scene(b.desc())
    rays = T.random_rays(200000, seed=9, box=(-2.0, 2.0))
    want, _ = oracle.trace(b.arrays(), rays, threads=8)
    want_any = sc.trace_host(rays, any_hit=True, cfg=BVH2)
    rb = N.DeviceBuffer.from_array(rays)
    hb, ha = N.DeviceBuffer(16 * len(rays)), N.DeviceBuffer(16 * len(rays))
    untouched = np.full(4 * len(rays), 7, np.int32)
    for n in (0, 1, 61, 5000, LARGEST, LARGEST + 5, len(rays)):
        cnt = N.DeviceBuffer.from_array(np.array([n], np.int32))
        hb.upload(untouched)
        N.check(N.lib.imba_intersect_dev(sc.h, rb.ptr, hb.ptr, len(rays), cnt.ptr, None, None), "intersect_dev")
        got = hb.download(N.HIT_DTYPE, len(rays))
        assert _same(got[:n], want[:n]) and (np.ascontiguousarray(got[n:]).view(np.int32) == 7).all(), n
        # two closest queues and an any-hit queue of the same rays
        k = n // 3
        batch = S.TraceBatch([(sc, rb, hb, k, None, False), (sc, rb.at(32 * k), hb.at(16 * k), len(rays) - k, cnt, False),
                              (sc, rb, ha, n, None, True)])
        left = min(n, len(rays) - k)
        for cfg in (None, Q4):
            hb.upload(untouched)
            batch.launch(cfg)
            got = hb.download(N.HIT_DTYPE, len(rays))
            assert _same(got[:k + left], want[:k + left]), (n, cfg)
            got_any = ha.download(N.HIT_DTYPE, len(rays))[:n]
            if cfg is None:
                assert _same(got_any, want_any[:n]), n
            else:
                assert np.array_equal(got_any["tri_id"] >= 0, want_any[:n]["tri_id"] >= 0), n
    assert sc.error_count() == 0


def test_recorded_batch(gpu):
    """A batch recorded into a graph after one plain launch, with the open choice of tree and with
    the quantized one: replays follow the queue sizes of later updates on both sides of the
    largest small queue.  The scene's stack is deeper than the LDS part."""
    b = T.random_tri_scene(200000, N.BUILDER_BINNED_SAH)[0]
    sc = S.Scene(b.desc())
    rays = T.random_rays(LARGEST + 3000, seed=10)
    want = sc.trace_host(rays, cfg=BVH2)
    assert sc.stack_depths(rays, cfg=Q4)[17:].sum() > 0
    rb, hb = N.DeviceBuffer.from_array(rays), N.DeviceBuffer(16 * len(rays))
    for cfg in (None, Q4):
        st = N.Stream()
        batch = S.TraceBatch([(sc, rb, hb, 500, None, False)])
        batch.launch(cfg, st)
        st.sync()
        S.Graph.begin(st)
        try:
            batch.launch(cfg, st)
        finally:
            g = S.Graph.end(st)
        for n in (500, len(rays), 77, LARGEST):
            batch.update([(sc, rb, hb, n, None, False)], st)
            hb.upload(np.full(4 * len(rays), 7, np.int32), st)
            g.launch(st)
            st.sync()
            got = hb.download(N.HIT_DTYPE, len(rays))
            assert _same(got[:n], want[:n]) and (np.ascontiguousarray(got[n:]).view(np.int32) == 7).all(), (n, cfg)


def test_spill_is_sized_for_one_lane_per_ray(gpu):
    """The launch of a small queue has four threads per ray, and its spill stack those of one lane per
    ray: a strided launch on a stream leaves room enough to record the small queue's.
    A device count on either side of the largest small queue then finds its place in it."""
    b = T.random_tri_scene(200000, N.BUILDER_BINNED_SAH)[0]
    sc = S.Scene(b.desc())
    assert S.wide_tree(b.arrays())["max_stack"] > 16
    for cap in (20000, LARGEST + 20000):
        rays = T.random_rays(cap, seed=12)
        want = sc.trace_host(rays, cfg=ONE_LANE)
        rb, hb, st = N.DeviceBuffer.from_array(rays), N.DeviceBuffer(16 * cap), N.Stream()
        cnt = N.DeviceBuffer.from_array(np.array([cap], np.int32))
        # eight blocks per CU: one thread per ray here, so the spill of one lane per ray
        strided = N.TraceConfig(256, 16, 0, 8, 4, 1, 0)
        sc.intersect(rb, hb, cap, strided, st)
        st.sync()
        S.Graph.begin(st)
        try:
            N.check(N.lib.imba_intersect_dev(sc.h, rb.ptr, hb.ptr, cap, cnt.ptr, N.C.byref(Q4), st.handle), "intersect_dev")
        finally:
            g = S.Graph.end(st)
        for n in (cap, 77, min(cap, LARGEST + 1), cap):
            cnt.upload(np.array([n], np.int32))
            hb.upload(np.full(4 * cap, 7, np.int32))
            g.launch(st)
            st.sync()
            got = hb.download(N.HIT_DTYPE, cap)
            assert _same(got[:n], want[:n]) and (np.ascontiguousarray(got[n:]).view(np.int32) == 7).all(), (cap, n)
    assert sc.error_count() == 0


@pytest.mark.parametrize("name", ["boxes", "sphere", "decal"])
def test_where_triangles_meet(gpu, name):
    """Where triangles meet or overlap the quantized tree's hits are its own (boxes are culled by rounded
    distances), and the same for every mapping of rays to lanes."""
    if name == "boxes":
        b, rays = T.box_scene(), T.random_rays(LARGEST + 5000, seed=3, box=(0.0, 2.2))
    else:
        b, points = T.sphere_scene() if name == "sphere" else T.decal_scene()
        rays = T.aimed_rays(points, LARGEST + 5000, seed=5)
    sc = S.Scene(b.desc())
    for any_hit in (False, True):
        want = sc.trace_host(rays, any_hit=any_hit, cfg=ONE_LANE)
        for n in (1000, LARGEST, len(rays)):
            assert _same(sc.trace_host(rays[:n], any_hit=any_hit, cfg=Q4), want[:n]), n
            assert _same(sc.trace_host(rays[:n], any_hit=any_hit, cfg=STRIDED), want[:n]), n
        if not any_hit:
            assert not _same(want, sc.trace_host(rays))  # the rays find such places
    assert sc.error_count() == 0
