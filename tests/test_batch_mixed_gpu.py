"""A batch whose streams differ in the luma search (transform types, depths or
neither): their frames share the rounds and their intra phases take different
kernels; equal to each stream's own sequence driver."""
import pytest

import mav1hip
import synth
from test_batch_gpu import check_against_sequences

pytestmark = pytest.mark.gpu


def test_batch_mixed_luma_search(gpu):
    opts = [dict(tx_search=0, tx_depth=0), dict(tx_search=1, tx_depth=0), dict(tx_search=0, tx_depth=1)]
    print("[batch] 3 x 142x98 full search, tx_search / tx_depth 0/0, 1/0, 0/1", flush=True)
    cfgs = []
    for o in opts:
        cfg = mav1hip.default_config(142, 98, turbo=0, qindex=110, keyint=60, altref=2)
        for k, v in o.items():
            setattr(cfg, k, v)
        cfgs.append(cfg)
    planes = [[synth.Synth(142, 98, 5 + i, n_objects=5, max_vel=9, noise_sigma=3.0).frame(t) for t in range(4)]
              for i in range(3)]
    check_against_sequences(cfgs, planes)
