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
