"""The node search's windows: full-pel radii below, at and past what the LDS
windows hold (32), with and without the decimated first stage, sub-pel costs
from the quarter-pel planes and from predictions, on frames whose last blocks
hang over the edges, of even and odd sizes; fields bit-exact against the oracle."""
import numpy as np
import pytest

import libs
import mav1hip

pytestmark = pytest.mark.gpu


def check(w, h, seed, cfg, fp):
    geo, frames = libs.make_sequence(w, h, 3, seed, n_objects=6, max_vel=20)
    ctx = mav1hip.Context(cfg)
    try:
        mv, mvg = ctx.motion_search(fp, frames[1], frames[0], frames[2])
        mo, go = libs.Impl("oracle").motion_search(fp, frames[1], frames[0], frames[2])
        assert np.array_equal(mv, mo), np.nonzero(mv != mo)[0][:8]
        if go is not None:
            assert np.array_equal(mvg, go), np.nonzero(mvg != go)[0][:8]
    finally:
        ctx.close()


@pytest.mark.parametrize("me_range", [4, 8, 20, 32, 40, 72])
@pytest.mark.parametrize("dec", [0, 1])
@pytest.mark.parametrize("w,h", [(142, 98), (141, 99)])
def test_turbo_ranges(gpu, w, h, me_range, dec):
    print(f"[me] {w}x{h} range {me_range} decimated {dec}", flush=True)
    mask = 0x47CBF1 | 0x20 if dec else 0x47CBF1 & ~0x20  # MAV1_T_ME_DEC
    cfg, fp = libs.turbo_params(w, h, "arf", me_range=me_range, knob_turbo_mask=mask)
    assert fp.me_range == me_range
    check(w, h, me_range, cfg, fp)


@pytest.mark.parametrize("w,h,me_range", [(66, 34, 8), (67, 35, 8), (142, 98, 32), (141, 99, 36), (142, 98, 36), (70, 130, 17)])
def test_full_search_ranges(gpu, w, h, me_range):
    print(f"[me] full search {w}x{h} range {me_range}", flush=True)
    cfg = mav1hip.default_config(w, h, turbo=0, qindex=100, me_range=me_range, multi_ref=1)
    fp, _ = mav1hip.setup_params(cfg, mav1hip.frame_info(order_hint=1, gold_differs=1))
    check(w, h, w + h, cfg, fp)
