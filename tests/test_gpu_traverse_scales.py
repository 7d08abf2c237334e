"""Closest and any hits on the MI355X against the oracle's brute force where
the BVH8's quantised boxes are tightest against rounding: very small and very
large triangles, geometry far from the origin, flat geometry, rays from far
away, along the axes (zero and negative-zero components) and with long
directions.  Hits are bit-identical, except that of overlapping triangles in
one plane, which a ray meets at distances that differ in their last bits,
either may be found."""
import struct
import tempfile
from pathlib import Path

import numpy as np
import pytest

import vision_amd as va
from oracle import oracle
from vision_amd import scenegen

pytestmark = pytest.mark.gpu

MISS = 0xFFFFFFFF


def _scene(tri, folder):
    n = len(tri) // 3
    fn = Path(folder) / "soup.vsmesh"
    idx = np.arange(3 * n, dtype=np.uint32)
    fn.write_bytes(b"VSMESH01" + struct.pack("<III", 3 * n, n, 0) + tri.astype(np.float32).tobytes() + idx.tobytes())
    s = scenegen.cornell_box(8, 8)
    s["shapes"] = [x for x in s["shapes"] if x["name"] == "light"]
    s["shapes"].append({"type": "model", "name": "soup", "param": {"fn": "soup.vsmesh", "material": "Gray"}})
    return s


@pytest.mark.parametrize("scale,offset,flat", [(1e-3, 0.0, False), (1.0, 300.0, False), (1e4, 0.0, False),
                                               (1.0, 0.0, True), (0.02, 50.0, True)])
def test_hits_equal_brute_force(gpu_ctx, scale, offset, flat):
    rng = np.random.default_rng(17)
    n = 3000
    tri = (rng.random((n, 1, 3)) * 2 - 1) + rng.normal(scale=0.05, size=(n, 3, 3))
    if flat:
        tri[..., 1] = 0.25
    tri = tri * scale + offset
    with tempfile.TemporaryDirectory() as d:
        sc = gpu_ctx.load_text(_scene(tri.reshape(-1, 3), d), base_dir=d)
        sc.build_accel()
    ex = sc.export()
    P, T = ex["positions"], ex["triangles"]
    m = 24000
    rays = np.zeros(m, va.RAY_DTYPE)
    # a third from inside, a third from 300 extents away, a third along an axis
    target = P[T[rng.integers(0, len(T), m), 0]] * 0.7 + P[T[rng.integers(0, len(T), m), 1]] * 0.3
    away = rng.normal(size=(m, 3))
    away /= np.linalg.norm(away, axis=1, keepdims=True)
    dist = np.where(np.arange(m) % 3 == 1, 300.0, 1.0)[:, None] * scale
    org = (target + away * dist).astype(np.float32)
    d = (target - org).astype(np.float32)
    axis = np.arange(m) % 3 == 2
    a = rng.integers(0, 3, m)
    along = np.where(rng.random((m, 3)) < 0.5, np.float32(0.0), np.float32(-0.0)).astype(np.float32)
    along[np.arange(m), a] = np.where(rng.random(m) < 0.5, -1.0, 1.0) * scale
    d[axis] = along[axis]
    org[axis] = (target - along * 3)[axis]
    rays["org"], rays["dir"], rays["t_max"] = org, d, np.finfo(np.float32).max
    flat_rays = np.concatenate([rays["org"], rays["t_min"][:, None], rays["dir"], rays["t_max"][:, None]], 1)
    hits = sc.trace_closest(rays)
    tri_id, t, _ = oracle.trace(P, T, flat_rays, bvh=False)
    hit = tri_id != MISS
    assert hit.mean() > 0.2
    assert np.array_equal(hits["tri"] != MISS, hit)
    assert flat or np.array_equal(hits["tri"], tri_id)
    if flat:
        # an ulp of each of the distance's sums and products
        np.testing.assert_allclose(hits["t"][hit], t[hit], rtol=1e-6)
    else:
        assert np.array_equal(hits["t"][hit], t[hit])
    rays["t_max"] = np.where(hit, hits["t"] * np.float32(0.999), 1.0).astype(np.float32)
    flat_rays[:, 7] = rays["t_max"]
    occ = sc.trace_any(rays)
    any_id, _, _ = oracle.trace(P, T, flat_rays, any_hit=True, bvh=False)
    assert np.array_equal(occ.astype(bool), any_id != MISS)
    sc.close()


@pytest.mark.parametrize("extent,size", [(4e21, 1e4), (1e25, 1e3), (3e33, 1.0)])
def test_hits_over_the_builder_extents(gpu_ctx, wide_soup, extent, size):
    """Extents at which a node's step is held as a NaN (from 2^65 on)."""
    P, _, flat_rays = wide_soup(extent, size)
    with tempfile.TemporaryDirectory() as d:
        sc = gpu_ctx.load_text(_scene(P, d), base_dir=d)
        sc.build_accel()
    ex = sc.export()
    rays = np.zeros(len(flat_rays), va.RAY_DTYPE)
    rays["org"], rays["t_min"], rays["dir"], rays["t_max"] = (flat_rays[:, 0:3], flat_rays[:, 3], flat_rays[:, 4:7],
                                                              flat_rays[:, 7])
    tri_id, t, _ = oracle.trace(ex["positions"], ex["triangles"], flat_rays, bvh=False)
    hit = tri_id != MISS
    assert hit.mean() > 0.1
    hits = sc.trace_closest(rays)
    assert np.array_equal(hits["tri"], tri_id)
    assert np.array_equal(hits["t"][hit], t[hit])
    assert np.array_equal(sc.trace_any(rays).astype(bool), hit)
    sc.close()
