"""The luma transform type / depth search of small intra blocks as a dataflow
of two-wave teams (csrc/recon_intra.h) against the oracle, bit-exact: depth
and type search in every combination, blocks that cross the frame's right and
bottom edge (sizes that are multiples of 8 but not of 16), smooth content
(larger intra blocks between the small ones) and noisy content (8x8 blocks),
low and high quantisers; and a batch whose streams differ in the search."""
import numpy as np
import pytest

import libs
import mav1hip
import synth
from test_batch_gpu import check_against_sequences
from test_recon_gpu import _check

pytestmark = pytest.mark.gpu


def _key(w, h, seed, q, noise, **kw):
    cfg = mav1hip.default_config(w, h, turbo=0, qindex=q, tile_cols_log2=1, **kw)
    fp, _ = mav1hip.setup_params(cfg, mav1hip.turbo_frame("key", 0))
    _, frames = libs.make_sequence(w, h, 3, seed, n_objects=8, max_vel=10, noise_sigma=noise)
    zero = np.zeros(fp.sb_cols * fp.sb_rows * 170, np.int32)
    _, _, blocks, sbs = libs.Impl("oracle").analyze(fp, frames[1], frames[0], frames[2], zero, zero)
    return cfg, fp, frames, blocks, sbs


@pytest.mark.parametrize("w,h", [(136, 104), (200, 136), (72, 88)])
@pytest.mark.parametrize("search,depth", [(1, 1), (1, 0), (0, 1)])
@pytest.mark.parametrize("q,noise", [(40, 0.5), (125, 3.0), (215, 6.0)])
def test_small_intra_search(gpu, w, h, search, depth, q, noise):
    print(f"\n[search] {w}x{h} tx_search {search} tx_depth {depth} q {q} noise {noise}", flush=True)
    cfg, fp, frames, blocks, sbs = _key(w, h, w + q, q, noise, tx_search=search, tx_depth=depth)
    _check(cfg, fp, frames, blocks, sbs)
    forced, _, _ = libs.force_intra_modes(fp, blocks, sbs, q)
    _check(cfg, fp, frames, forced, sbs)


def test_batch_with_and_without_search(gpu):
    print("\n[search] batch: 200x136 full RD altref 2 + 200x136 turbo", flush=True)
    cfgs = [mav1hip.default_config(200, 136, turbo=0, qindex=125, altref=2, leaf=1, tile_cols_log2=1),
            mav1hip.default_config(200, 136, turbo=1, qindex=125, restoration=1)]
    planes = [[synth.Synth(200, 136, 50 + i, n_objects=4, max_vel=8, noise_sigma=2.0).frame(t) for t in range(5)]
              for i in range(2)]
    check_against_sequences(cfgs, planes)
