"""The restoration search on synthetic planes at the sizes where its split
into column tasks, fit chunks and 4x4 blocks has remainders: units of one
column of tasks to the largest unit (95 x 103), odd chroma sizes, one to five
stripe segments per unit, more blocks and tasks than threads. The source is
the filtered frame blurred and with noise, so that Wiener and self-guided
filters win and the references change from unit to unit."""
import numpy as np
import pytest

import libs
import mav1hip

pytestmark = pytest.mark.gpu

CASES = [  # w, h, noise, lr_test, q
    (16, 16, 6, 0, 125),
    (34, 18, 0, 0, 60),
    (70, 58, 10, 1, 125),
    (94, 158, 4, 0, 200),      # one unit of 94 x 87 after the first 56 rows; chroma 47 x 79
    (158, 94, 12, 0, 125),     # last unit 94 wide; 94 rows in one unit
    (222, 166, 3, 1, 90),
    (190, 190, 20, 0, 255),
    (318, 286, 8, 0, 40),
]


def planes(fp, n, noise, seed):
    """Source, CDEF output and deblocked frames of n bytes in the padded layout."""
    rng = np.random.default_rng(seed)
    cdef, dbk, src = (np.zeros(n, np.uint8) for _ in range(3))
    for p in range(3):
        w, h = (fp.frame_w + (p > 0)) >> (p > 0), (fp.frame_h + (p > 0)) >> (p > 0)
        yy, xx = np.mgrid[0:h, 0:w]
        base = 128 + 70 * np.sin(xx / (5.0 + p)) * np.cos(yy / 7.0) + 40 * ((xx // 13 + yy // 11) & 1)
        s = np.clip(base, 0, 255)
        c = s + rng.normal(0, noise, s.shape)
        c[:, 1:] = 0.6 * c[:, 1:] + 0.4 * c[:, :-1]
        d = c + rng.normal(0, 2, s.shape)
        for a, v in ((cdef, c), (dbk, d), (src, s)):
            idx = fp.offset[p] + np.arange(h)[:, None] * fp.stride[p] + np.arange(w)[None]
            a[idx] = np.clip(np.rint(v), 0, 255).astype(np.uint8)
    return src, cdef, dbk


@pytest.mark.parametrize("w,h,noise,lr_test,q", CASES)
def test_lr_search_edges_equal_oracle(gpu, w, h, noise, lr_test, q):
    cfg = mav1hip.default_config(w, h, turbo=1, qindex=q, restoration=1)
    fp, _ = mav1hip.setup_params(cfg, mav1hip.turbo_frame("arf", 1))
    ctx = mav1hip.Context(cfg)
    try:
        src, cdef, dbk = planes(fp, ctx.frame_bytes, noise, w * 1000 + h)
        print(f"[lr search] {w}x{h} noise {noise} lr_test {lr_test} q{q}", flush=True)
        uo, to = libs.Filters("oracle").lr_select(fp, src, cdef, dbk, lr_test)
        for _ in range(2):
            ug, tg, _ = ctx.lr_select(fp, src, cdef, dbk, lr_test)
            assert tg == to
            bad = np.nonzero((ug != uo).any(axis=1))[0]
            assert bad.size == 0, f"units differ at {bad[:8]}: {ug[bad[:2]]} {uo[bad[:2]]}"
    finally:
        ctx.close()
