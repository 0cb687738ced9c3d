"""Cache frames whose update jobs run in the frame's own bounces (the default,
rtx_tuning.cacheUpkeep 1), with what such a frame may combine: lookups alone,
ADRRS roulette without splitting, guided directions, and both.  The image and
the cache are those of the frame with every job after it (cacheUpkeep 2), bit
for bit, and the paths of that are the oracle's (bars as in test_gpu_adrrs)."""
import numpy as np
import pytest

import rtxamd
import scenes
from oracle.binding import OracleScene
from parity import check_paths
from rtxamd import abi
from test_gpu_guiding import regions_and_mixtures
from test_gpu_icache import cornell_state

pytestmark = pytest.mark.gpu

W, H = 72, 50  # no whole number of waves


@pytest.fixture(scope="module")
def cornell():
    hs = rtxamd.HostScene.generate(abi.SCENE_CORNELL)
    orc = OracleScene(abi, hs.desc())
    return hs, orc, cornell_state(orc, hs)


@pytest.mark.parametrize("adrrs,guide", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_merged_frames_equal_frames_with_jobs_after(renderer, cornell, adrrs, guide):
    hs, orc, st0 = cornell
    est = np.full((W * H, 4), 0.05, np.float32)
    renderer.estimate_write(est, W, H)
    orc.estimate_set(est, W, H)
    regions, vmms = regions_and_mixtures(0)
    if guide:
        renderer.guiding_set(regions, vmms)
        orc.guiding_set(regions, vmms)
    ds = renderer.upload(hs)

    def frame(mode, flags=0, **kw):
        kw = dict(dict(useADRRS=adrrs, adrrsS=2.0), **kw)
        fp = scenes.params(hs, W, H, 1, maxDepth=8, enableMIS=1, useIrradianceCache=1, irradianceCreateProb=0.01,
                           irradianceUpdateProb=0.02, adrrsSplit=0, useGuiding=guide, guidingProb=0.5,
                           sample_offset=7, flags=abi.RTX_FRAME_RESET_ACCUM | flags, **kw)
        renderer.set_tuning(cacheUpkeep=mode)
        renderer.ic_create(st0.max_entries)
        renderer.ic_write(st0)
        renderer.render(ds, fp)
        return fp, renderer.ic_read(), renderer.read_image(W, H)

    try:
        fp, s_keep, i_keep = frame(2, abi.RTX_FRAME_KEEP_PATHS)
        rgb, sig = renderer.read_paths(W * H)
        after, merged = frame(2), frame(1)
        no_adrrs = frame(1, useADRRS=0)
    finally:
        renderer.set_tuning(cacheUpkeep=1)
        renderer.guiding_set([], [])
        ds.close()
    orgb, osig = orc.ic_frame(fp, st0.copy())[:2]
    f32 = orc.ic_frame(fp, st0.copy(), prec=32)[:2]
    check_paths(f"cache frame, ADRRS {adrrs}, guiding {guide}", rgb, sig, orgb, osig, f32, abs_same=0.95,
                abs_within=0.99)
    # the comparison is of something: updates ran, and ADRRS changes the image
    assert (merged[1].entries["numUpdates"][:st0.count] > st0.entries["numUpdates"][:st0.count]).sum() > 20
    assert ((merged[2] != no_adrrs[2]).any(-1).mean() > 0.1) == bool(adrrs)
    for _, s, i in (after, merged):
        assert np.array_equal(i.view(np.uint32), i_keep.view(np.uint32))
        assert (s.hdr.nextCacheSlot, s.hdr.nextUpdateSlot) == (s_keep.hdr.nextCacheSlot, s_keep.hdr.nextUpdateSlot)
        assert s.entries.tobytes() == s_keep.entries.tobytes() and s.spheres.tobytes() == s_keep.spheres.tobytes()
