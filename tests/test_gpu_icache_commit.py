"""Committing a frame's cache jobs side by side against the oracle's job by job
commit of the same results: updates that meet every record at most once and
(more elections than records) several times, creations that fill the cache to
its last slot, and more creations than one block takes at a time."""
import numpy as np
import pytest

import rtxamd
import scenes
from oracle.binding import OracleScene, ic_apply
from rtxamd import abi
from test_gpu_icache import cornell_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entries,frames,size,create,update", [
    (3000, 4, 64, 0.02, 0.01),    # few elections: one update a record
    (40, 1, 64, 0.02, 0.2),       # more elections than records, no free slot left
    (700, 2, 64, 0.5, 0.005),     # creations run into the last slot
    (20000, 1, 128, 0.9, 0.001),  # more than 1024 creations
])
def test_commit_matches_job_order(renderer, entries, frames, size, create, update):
    hs = rtxamd.HostScene.generate(abi.SCENE_CORNELL)
    st0 = cornell_state(OracleScene(abi, hs.desc()), hs, frames=frames, max_entries=entries)
    renderer.ic_create(entries)
    renderer.ic_write(st0)
    fp = scenes.params(hs, size, size, 1, maxDepth=8, enableMIS=1, useIrradianceCache=1, irradianceCreateProb=create,
                       irradianceUpdateProb=update, sample_offset=9,
                       flags=abi.RTX_FRAME_KEEP_PATHS | abi.RTX_FRAME_RESET_ACCUM)
    ds = renderer.upload(hs)
    try:
        renderer.render(ds, fp)
    finally:
        ds.close()
    jobs, sub, _ = renderer.ic_read_jobs()
    got = renderer.ic_read()
    ref = st0.copy()
    ic_apply(abi, fp, ref, jobs, sub, prec=32)
    c = ref.count
    assert len(jobs) > 0 and got.count == c
    assert np.array_equal(ref.entries["numUpdates"][:c], got.entries["numUpdates"][:c])
    assert np.allclose(got.spheres["center"][:c], ref.spheres["center"][:c], rtol=0, atol=1e-6)
    assert np.allclose(got.entries["normal"][:c], ref.entries["normal"][:c], rtol=0, atol=1e-6)
    # a mean of at most 200 positive terms, in both the same order: rounding below 200 x 2^-24 = 1.2e-5
    for a, b in ((got.entries["harmonicR"], ref.entries["harmonicR"]), (got.spheres["radius"], ref.spheres["radius"])):
        assert (b[:c] > 0).all() and np.allclose(a[:c], b[:c], rtol=1.2e-5, atol=0)
    assert (got.hdr.nextCacheSlot, got.hdr.maxCaches) == (ref.hdr.nextCacheSlot, ref.hdr.maxCaches)
    for f in ("color", "rotGrad", "transGrad"):
        a, b = got.entries[f][:c].astype(np.float64), ref.entries[f][:c].astype(np.float64)
        # 1e-4 of the record's scale.  A gradient is a sum of up to 400 signed
        # terms, whose rounding is bounded by 400 x 2^-24 = 2.4e-5 of their
        # absolute sum: records whose terms cancel to less than a quarter of
        # that may exceed the bar, one in a thousand allowed
        ok = (np.abs(a - b) <= 1e-4 * np.maximum(np.abs(b).max(1, keepdims=True), 1e-6)).all(1)
        assert ok.all() if f == "color" else (~ok).sum() <= len(ok) // 1000, f
