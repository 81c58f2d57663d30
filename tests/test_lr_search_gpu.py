"""The restoration search on synthetic planes at the sizes where its split
into column tasks, fit chunks and 4x4 blocks has remainders: units of one
column of tasks to the largest unit (95 x 103), odd luma and chroma sizes, one
to four stripe segments per unit, more blocks and tasks than threads. From
unit to unit the filtered frame is the source blurred (a Wiener filter wins),
edges with noise (a self-guided set wins) or nearly the source, so that the
references change between the units; the forced pattern takes both filters at
every size."""
import numpy as np
import pytest

import libs
import mav1hip
import synth

CASES = [  # w, h, noise, kind of the first unit, q
    (16, 16, 6, 1, 20),
    (17, 19, 6, 1, 60),
    (34, 18, 6, 0, 20),
    (70, 58, 4, 0, 20),
    (71, 57, 6, 1, 60),
    (95, 159, 6, 0, 60),       # the second unit is the largest, 95 x 103, with edges and noise; chroma 48 x 80
    (95, 159, 6, 2, 60),       # the same unit blurred
    (159, 95, 6, 0, 60),       # 95 columns behind 64; 95 rows in one unit
    (222, 166, 4, 1, 60),
    (191, 190, 9, 0, 40),
    (317, 318, 5, 0, 40),      # chroma 159 x 159: the last unit 95 x 99 in four segments
    (317, 318, 5, 2, 40),      # ... blurred in U
]


def planes(fp, noise, first, seed):
    """Source, CDEF output and deblocked frames in the padded layout."""
    geo = synth.Geometry(fp.frame_w, fp.frame_h)
    rng = np.random.default_rng(seed)
    cdef, dbk, src = (np.zeros(geo.frame_bytes, np.uint8) for _ in range(3))
    for p in range(3):
        w, h = (fp.frame_w + (p > 0)) >> (p > 0), (fp.frame_h + (p > 0)) >> (p > 0)
        yy, xx = np.mgrid[0:h, 0:w]
        rows, cols = fp.lr_unit_rows[p], fp.lr_unit_cols[p]
        unit = np.minimum(yy // 64, rows - 1) * cols + np.minimum(xx // 64, cols - 1) + first + p
        wave = np.clip(128 + 70 * np.sin(xx / (5.0 + p)) * np.cos(yy / 7.0) + 40 * ((xx // 13 + yy // 11) & 1), 0, 255)
        blur = wave.copy()
        blur[:, 1:] = 0.6 * wave[:, 1:] + 0.4 * wave[:, :-1]
        blur[1:] = 0.7 * blur[1:] + 0.3 * blur[:-1]
        edges = 98.0 + 60 * ((xx // 16 + yy // 16) & 1)
        sigma = np.select([unit % 3 == 0, unit % 3 == 1], [1.0, noise * np.array([0.5, 1, 2])[unit // 3 % 3]], 0.4)
        s = np.where(unit % 3 == 1, edges, wave)
        c = np.select([unit % 3 == 0, unit % 3 == 1], [blur, edges], wave) + sigma * rng.normal(0, 1, s.shape)
        d = c + rng.normal(0, 2, s.shape)
        for a, v in ((cdef, c), (dbk, d), (src, s)):
            idx = fp.offset[p] + np.arange(h)[:, None] * fp.stride[p] + np.arange(w)[None]
            a[idx] = np.clip(np.rint(v), 0, 255).astype(np.uint8)
    return src, cdef, dbk


def case(w, h, noise, first, q, lr_test):
    """Parameters, planes and the oracle's units and types."""
    cfg = mav1hip.default_config(w, h, turbo=1, qindex=q, restoration=1)
    fp, _ = mav1hip.setup_params(cfg, mav1hip.turbo_frame("arf", 1))
    src, cdef, dbk = planes(fp, noise, first, w * 1000 + h)
    return cfg, fp, src, cdef, dbk, libs.Filters("oracle").lr_select(fp, src, cdef, dbk, lr_test)


def test_cases_decide_both_filters():
    """The oracle's choices: no case leaves every unit alone, both filters win
    in luma and chroma and on the largest unit, with different sets, and the
    forced pattern takes the largest unit's sets, too."""
    wins = {False: set(), True: set()}
    largest, sets = set(), set()
    for c in CASES:
        _, fp, _, _, _, (u, types) = case(*c, lr_test=0)
        assert any(types), f"{c}: nothing restored"
        for k in np.nonzero(u[:, 0])[0]:
            wins[bool(k >= fp.lr_unit_off[1])].add(int(u[k, 0]))
        forced = case(*c, lr_test=1)[5][0]
        sets |= {int(k[1]) for k in np.concatenate([u, forced]) if k[0] == 2}
        if c[:2] == (95, 159):
            largest.add(int(u[1, 0]))
            assert forced[1, 0] == 2
    assert wins[False] == wins[True] == largest == {1, 2}
    assert len(sets) >= 4, sets


@pytest.mark.gpu
@pytest.mark.parametrize("lr_test", [0, 1])
@pytest.mark.parametrize("w,h,noise,first,q", CASES)
def test_lr_search_edges_equal_oracle(gpu, w, h, noise, first, q, lr_test):
    print(f"[lr search] {w}x{h} noise {noise} first {first} lr_test {lr_test} q{q}", flush=True)
    cfg, fp, src, cdef, dbk, (uo, to) = case(w, h, noise, first, q, lr_test)
    assert any(to)
    ctx = mav1hip.Context(cfg)
    try:
        for _ in range(2):
            ug, tg, _ = ctx.lr_select(fp, src, cdef, dbk, lr_test)
            assert tg == to
            bad = np.nonzero((ug != uo).any(axis=1))[0]
            assert bad.size == 0, f"units differ at {bad[:8]}: {ug[bad[:2]]} {uo[bad[:2]]}"
    finally:
        ctx.close()
