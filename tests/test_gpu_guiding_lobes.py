"""The guiding update's sample sums on the device are built for 8, 16 and 32
lobes, and its region segments come from the sorted samples: each lobe limit
at the edges of those builds, and one region as well as many (some of them
empty), against the oracle's update of the same records."""
import numpy as np
import pytest

import rtxamd
import scenes
from oracle.binding import OracleGuide
from parity import log
from rtxamd import abi
from test_gpu_guiding import fib_sphere, mixture_pdf_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits,lobes", [(0, 8), (2, 9), (3, 16), (5, 17), (3, 32)])
def test_update_at_every_lobe_limit(renderer, splits, lobes):
    hs = rtxamd.HostScene.generate(abi.SCENE_CORNELL)
    ds = renderer.upload(hs)
    box = ds.bounds()
    # thresholds low enough that lobes split towards the limit within two updates
    opts = abi.guiding_options(maxComponents=lobes, minSamplesForSplitting=64, minSamplesForPostSplitFitting=64,
                               minSamplesForMerging=256, splitMinDivergence=0.05)
    renderer.set_guiding_options(opts)
    renderer.guiding_init(box, splits, parallax=True)
    og, o32 = (OracleGuide(abi, box, splits, parallax=True, prec=p, options=opts) for p in (64, 32))
    dirs = fib_sphere(2000)
    try:
        for frame in range(2):
            renderer.render(ds, scenes.params(hs, 96, 96, 1, maxDepth=6, enableMIS=1, updateGuiding=1,
                                              useGuiding=int(frame > 0), sample_offset=frame))
            dd = renderer.guiding_read_samples(96, 96)
            og.update(dd)
            o32.update(dd)
        _, gv = renderer.guiding_get_wide()
        _, ov = og.regions_wide()
        _, fv = o32.regions_wide()
        used = [v.usedDistributions for v in gv]
        errs, errs32 = [], []
        for r in range(len(gv)):
            if (dd["flags"] == r).sum() < 50:
                continue
            x = np.array(ov[r].meanPosition[:], np.float64)
            pg, po, pf = (mixture_pdf_grid(v[r], dirs, x) for v in (gv, ov, fv))
            errs.append(np.abs(pg - po).mean() / po.mean())
            errs32.append(np.abs(pf - po).mean() / po.mean())
        log(f"{len(gv)} regions, limit {lobes}: lobes {min(used)}..{max(used)}; density L1 vs FP64 median "
            f"{np.median(errs):.2e} max {max(errs):.2e}, FP32 oracle {np.median(errs32):.2e} {max(errs32):.2e}")
        assert max(used) <= lobes
        # the bars of test_guiding_update_matches_oracle_em: the FP32 oracle's own distance from FP64
        assert np.median(errs) <= max(1e-3, 2 * np.median(errs32))
        assert max(errs) <= max(0.05, 2 * max(errs32))
    finally:
        renderer.set_guiding_options()
        renderer.guiding_set([], [])
        ds.close()
