"""The persistent traversal's work distribution on the device: a launch
traces the same rays whatever its size, its static span, its chunks and the
lanes that are left over (librtxamd.so through the C ABI)."""
import numpy as np
import pytest

import rtxamd
from rtxamd import abi

pytestmark = pytest.mark.gpu

N = 200003


@pytest.fixture(scope="module")
def room():
    r = rtxamd.Renderer(0)
    ds = r.upload(rtxamd.HostScene.generate(abi.SCENE_ROOM, 3, 12512))
    rng = np.random.default_rng(7)
    d = rng.normal(size=(N, 3))
    rays = rtxamd.rays_array(rng.uniform((-9.9, 0.1, -9.9), (9.9, 9.9, 9.9), (N, 3)),
                             d / np.linalg.norm(d, axis=1, keepdims=True))
    # the same rays one small call after another: no wave of these fetches past its static slice
    parts = [r.trace_closest_noalloc(ds, rays[i:i + 4096]) for i in range(0, N, 4096)]
    yield r, ds, rays, [np.concatenate(c) for c in zip(*parts)]
    ds.close()
    r.close()


# one block a CU of 128 threads (two waves): a static span of 128 rays a CU, and
# slices of fewer than 64 rays below half of it, so these sizes end before, on
# and after those edges, within the first chunks and far past them
@pytest.mark.parametrize("n", ["1", "63", "65", "span//128-1", "span//128+1", "span//2-1", "span//2", "span//2+1",
                               "span-1", "span", "span+1", "span+65", "3*span+17", "all"])
def test_every_size_traces_the_same_rays(room, n):
    r, ds, rays, want = room
    import torch
    span = 128 * torch.cuda.get_device_properties(0).multi_processor_count
    n = min(N, eval(n, {"span": span, "all": N}))
    base = r.tuning().traceBlocksPerCU
    try:
        for blocks in (1, base):
            r.set_tuning(traceBlocksPerCU=blocks)
            got = r.trace_closest(ds, rays[:n])
            for a, b in zip(got, want):
                assert np.array_equal(a.view(np.uint32), b[:n].view(np.uint32))
            assert np.array_equal(r.trace_occluded(ds, rays[:n]) != 0, want[1][:n] >= 0)
    finally:
        r.set_tuning(traceBlocksPerCU=base)


def test_deep_tree_traces_like_brute_force(renderer):
    """Triangles over 60 nested scales, whose tree is 33 levels of nodes deep:
    closest hits equal those of every triangle tested in FP64, where no hit
    is within 1e-3 of an edge."""
    i = np.arange(60000)
    x = (4.0 ** -(i % 60) * np.where((i // 60) % 2, -1.0, 1.0)).astype(np.float32)
    tri = np.stack([np.stack([x, x, x], 1), np.stack([2 * x, x, x], 1), np.stack([x, 2 * x, x], 1)], 1)
    hs = rtxamd.HostScene.new()
    mat = hs.add_material(rtxamd.diffuse((0.5, 0.5, 0.5)))
    hs.add_mesh(tri.reshape(-1, 3), np.arange(3 * len(x), dtype=np.uint32).reshape(-1, 3), mat,
                normals=np.tile(np.float32([0, 0, 1]), (3 * len(x), 1)))
    hs.add_point_light((0.0, 0.0, 5.0), (1.0, 1.0, 1.0))
    hs.finalize()
    rng = np.random.default_rng(3)
    n = 256
    org = rng.normal(size=(n, 3))
    org = (4.0 * org / np.linalg.norm(org, axis=1, keepdims=True)).astype(np.float32)
    b = rng.dirichlet((2, 2, 2), n)
    at = (tri[rng.integers(0, 8, n) + 60 * rng.integers(0, 2, n)] * b[..., None]).sum(1)
    d = at - org
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    ds = renderer.upload(hs)
    try:
        assert ds.info().maxDepth > 21
        t, prim, _, _ = renderer.trace_closest(ds, rtxamd.rays_array(org, d))
        occ = renderer.trace_occluded(ds, rtxamd.rays_array(org, d))
    finally:
        ds.close()
    v = tri[:120].astype(np.float64)  # each scale and sign once: the others lie on these
    o, dd = org.astype(np.float64)[:, None], d.astype(np.float64)[:, None]
    tt = (v[None, :, 0, 2] - o[..., 2]) / dd[..., 2]  # every triangle lies in a plane of constant z
    h = o + tt[..., None] * dd
    u = ((h - v[None, :, 0]) / x[:120].astype(np.float64)[None, :, None])[..., :2]
    edge = np.minimum(u.min(-1), 1.0 - u.sum(-1))  # inside where positive
    inside = (edge > 0) & (tt >= 1e-3)
    clear = (np.abs(edge) > 1e-3).all(1)
    want = np.where(inside, tt, np.inf).min(1)
    assert clear.sum() > 150
    hit = np.isfinite(want)
    assert np.array_equal((prim >= 0)[clear], hit[clear]) and np.array_equal((occ != 0)[clear], hit[clear])
    assert np.allclose(t[clear & hit], want[clear & hit], rtol=1e-5)
