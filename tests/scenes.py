"""Seeded test scenes and ray sets shared by the tests (host side only)."""
from __future__ import annotations

import numpy as np

from imbatracer_amd import native as N
from imbatracer_amd import scene as S

from imbatracer_amd.workloads import C1_CAMERA, C1_LIGHT, primary_rays, random_tri_scene as _rts, shadow_rays  # noqa: F401


def random_tri_scene(n: int, builder=N.BUILDER_BINNED_SAH, seed: int = 0x1234):
    return _rts(n, builder, seed)


def random_rays(n: int, seed: int = 5, box=(-0.2, 1.2)) -> np.ndarray:
    """Incoherent rays: origins in a box around the unit cube, uniform directions."""
    rng = np.random.default_rng(seed)
    o = rng.uniform(box[0], box[1], (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=1, keepdims=True).astype(np.float32)
    return S.make_rays(o, d.astype(np.float32), np.float32(0.0), np.float32(3.4028235e38))


def rot(axis: int, angle: float) -> np.ndarray:
    c, s = np.cos(angle), np.sin(angle)
    m = np.eye(4, dtype=np.float64)
    a, b = [(1, 2), (0, 2), (0, 1)][axis]
    m[a, a], m[a, b], m[b, a], m[b, b] = c, -s, s, c
    return m


def instanced_scene(builder=N.BUILDER_SBVH):
    """Three meshes, seven instances with rotations, scales and translations."""
    b = S.SceneBuild()
    v0, i0 = S.random_triangles(600, 11)
    v1, i1 = S.icosphere(2, 0.3, (0.0, 0.0, 0.0), 1)
    v2, i2 = S.random_triangles(300, 12)
    i2[:, 3] = 2
    m0, m1, m2 = b.add_mesh(v0, i0), b.add_mesh(v1, i1), b.add_mesh(v2, i2)
    rng = np.random.default_rng(3)
    for k, m in enumerate([m0, m1, m2, m1, m0, m1, m2]):
        t = np.eye(4)
        t[:3, 3] = rng.uniform(-1.5, 1.5, 3)
        sc = np.diag([rng.uniform(0.5, 1.5)] * 3 + [1.0])
        mat = t @ rot(k % 3, rng.uniform(0, 6.28)) @ sc
        b.add_instance(m, mat.astype(np.float32))
    b.run(builder, 2)
    return b


def masked_scene():
    """Random triangles with texcoords and a checkerboard opacity mask on material 0."""
    v, i = S.random_triangles(3000, 21)
    rng = np.random.default_rng(4)
    tc = rng.random((len(v), 2), dtype=np.float32) * 3.0
    b = S.SceneBuild()
    b.add_mesh(v, i, tc)
    yy, xx = np.mgrid[0:8, 0:16]
    b.set_mask(0, ((xx + yy) % 2).astype(np.uint8))
    b.run(N.BUILDER_BINNED_SAH, 1)
    return b


def _mesh_scene(v, tri):
    """One mesh of points v (n, 3) and triangles tri (m, 3), binned SAH."""
    v4 = np.ones((len(v), 4), np.float32)
    v4[:, :3] = v
    i4 = np.zeros((len(tri), 4), np.uint32)
    i4[:, :3] = tri
    b = S.SceneBuild()
    b.add_mesh(v4, i4)
    b.run(N.BUILDER_BINNED_SAH, 1)
    return b


def aimed_rays(points, n: int, seed: int) -> np.ndarray:
    """Rays from a sphere of radius 4 towards points drawn from `points`."""
    rng = np.random.default_rng(seed)
    o = rng.normal(size=(n, 3))
    o = (4.0 * o / np.linalg.norm(o, axis=1, keepdims=True)).astype(np.float32)
    d = points[rng.integers(0, len(points), n)] - o
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    return S.make_rays(o, d, np.float32(0.0), np.float32(3.4028235e38))


def box_scene(n: int = 300, seed: int = 1):
    """Axis-aligned boxes on a coarse lattice: many faces are coplanar and overlap."""
    rng = np.random.default_rng(seed)
    lo, size = rng.integers(0, 16, (n, 3)), rng.integers(1, 5, (n, 3))
    corner = np.array([[c & 1, (c >> 1) & 1, c >> 2] for c in range(8)])
    v = (lo[:, None] + size[:, None] * corner).astype(np.float32) / 8
    quads = np.array([[0, 1, 3, 2], [4, 6, 7, 5], [0, 4, 5, 1], [2, 3, 7, 6], [0, 2, 6, 4], [1, 5, 7, 3]])
    tri = np.concatenate([quads[:, [0, 1, 2]], quads[:, [0, 2, 3]]])
    return _mesh_scene(v.reshape(-1, 3), np.concatenate([tri + 8 * k for k in range(n)]))


def sphere_scene():
    """An icosphere and its vertices (each shared by five or six triangles)."""
    v, i = S.icosphere(4, 1.0, (0.0, 0.0, 0.0), 1)
    return _mesh_scene(v[:, :3], i[:, :3]), v[:, :3]


def decal_scene():
    """A floor of 40 x 40 squares with a coplanar 7 x 7 decal on it, and their vertices."""
    def squares(n, lo, hi):
        g = np.linspace(lo, hi, n + 1)
        x, y = np.meshgrid(g, g)
        a = np.arange(n * (n + 1)).reshape(n, n + 1)[:, :n].ravel()
        tri = np.concatenate([np.stack([a, a + 1, a + n + 2], 1), np.stack([a, a + n + 2, a + n + 1], 1)])
        return np.stack([x.ravel(), y.ravel(), np.zeros(x.size)], 1).astype(np.float32), tri
    v0, t0 = squares(40, 0.0, 1.0)
    v1, t1 = squares(7, 0.25, 0.75)
    v = np.concatenate([v0, v1])
    return _mesh_scene(v, np.concatenate([t0, t1 + len(v0)])), v
