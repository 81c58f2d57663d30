"""Analysis items whose blocks have few 4x4 units or hang over the frame's
edge: odd block counts, all partitions (4:1 blocks with 4-tap chroma), every
angle, chroma from luma, one and two references and their average, at
quantisers that pick different candidates; equal to the oracle."""
import pytest

import libs
import mav1hip
from test_analysis_gpu import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,q", [(18, 34, 30), (67, 35, 60), (66, 34, 200), (142, 98, 90), (141, 99, 120), (98, 162, 255)])
@pytest.mark.parametrize("kind", ["key", "inter", "compound"])
def test_analysis_edges(gpu, w, h, q, kind):
    print(f"[analysis] {w}x{h} q{q} {kind}", flush=True)
    kw = dict(multi_ref=1, compound=1) if kind == "compound" else {}
    cfg = mav1hip.default_config(w, h, turbo=0, qindex=q, **kw)
    fr = mav1hip.turbo_frame("key", 0) if kind == "key" else mav1hip.frame_info(order_hint=1, gold_differs=1)
    fp, _ = mav1hip.setup_params(cfg, fr)
    geo, frames = libs.make_sequence(w, h, 3, w + q, n_objects=5, max_vel=9)
    run_case(cfg, fp, frames)
