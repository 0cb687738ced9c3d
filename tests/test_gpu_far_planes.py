"""Rays along an axis, exactly or nearly, over a ground so wide that the ray
parameters of its box planes overflow FP32: the ground is hit (librtxamd.so
through the C ABI; tests/native/bvh_ray_check.cpp checks the box test itself)."""
import numpy as np
import pytest

import rtxamd
import scenes
from rtxamd import abi

pytestmark = pytest.mark.gpu

N = 500


@pytest.mark.parametrize("half,tilt", [(1.0, 0.0), (100.0, 1e-37), (1000.0, 1e-36), (1000.0, 1e-40), (4e8, 0.0),
                                       (1e9, 0.0)])
def test_wide_ground_is_hit(renderer, half, tilt):
    hs = rtxamd.HostScene.new()
    mat = hs.add_material(rtxamd.diffuse((0.5, 0.5, 0.5)))
    p, i = scenes.quad((-half, -half, 0), (half, -half, 0), (half, half, 0), (-half, half, 0))
    hs.add_mesh(p, i, mat)
    hs.add_point_light((0.0, 0.0, half), (1.0, 1.0, 1.0))
    hs.finalize()
    rng = np.random.default_rng(1)
    org = rng.uniform(-0.9 * half, 0.9 * half, (N, 3)).astype(np.float32)
    d = np.zeros((N, 3), np.float32)
    d[:, :2] = rng.choice([tilt, -tilt], (N, 2))
    d[:, 2] = -np.sign(org[:, 2])
    rays = rtxamd.rays_array(org, d, tmax=1e10)
    ds = renderer.upload(hs)
    try:
        t, prim, _, _ = renderer.trace_closest(ds, rays)
        occ = renderer.trace_occluded(ds, rays)
    finally:
        ds.close()
    assert (prim >= 0).all() and (occ == 1).all()
    assert np.allclose(t, np.abs(org[:, 2]), rtol=1e-5)
