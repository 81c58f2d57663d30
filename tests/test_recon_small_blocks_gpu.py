"""Reconstruction of a caller's own blocks where a superblock holds blocks
below 8x8 and 4:1 blocks (which the analysis never chooses) between blocks of
8x8 .. 16x16: the latter run in the level schedule's segments, the former by
the whole workgroup, and BlockDecoded and the chroma cells that several blocks
share follow decode order. Bit-exact against the oracle, with random modes,
without and with a luma search, on odd frame sizes too."""
import numpy as np
import pytest

import libs
import mav1hip
from test_recon_gpu import _check, _setup

pytestmark = pytest.mark.gpu

# block sizes by (log2 width, log2 height) in 4x4 units
BSIZE = {(0, 0): 0, (0, 1): 1, (1, 0): 2, (1, 1): 3, (2, 2): 6, (3, 3): 9, (0, 2): 16, (2, 0): 17}
LOG2 = {v: k for k, v in BSIZE.items()}


def _split(b, lw, lh):
    """Intra block b cut into parts of (lw, lh): their records in decode
    order. Parts that share a chroma cell share its levels."""
    W, H = (1 << k for k in LOG2[int(b[2])])
    w, h = 1 << lw, 1 << lh
    out = []
    for n, (r, c) in enumerate((r, c) for r in range(0, H, h) for c in range(0, W, w)):
        p = b.copy()
        p[0], p[1], p[2] = b[0] + r, b[1] + c, BSIZE[lw, lh]
        p[14] = b[14] + n * w * h * 16
        cells = max(1, w >> 1) * max(1, h >> 1) * 16  # of the part's chroma
        at = (n >> (lw == 0 or lh == 0)) * cells if W * H > 4 else 0
        p[15], p[16] = b[15] + at, b[16] + at
        out.append(p)
    return out


def _cut(b, fp, rng, room):
    """Random cuts of intra block b down to 4x4, at most `room` more blocks.
    Not below 8x8 at the top of the frame and the left of a tile: a part at an
    odd row or column there has a neighbour, but its chroma, which starts at
    the even one, has none (the oracle reads before the plane)."""
    edge = b[0] == 0 or b[1] % (fp.tile_w_sb * 16) == 0
    kinds = {9: [(2, 2)], 6: [(1, 1)] + ([] if edge else [(1, 1), (0, 2), (2, 0)]),
             3: [] if edge else [(0, 0), (0, 1), (1, 0)]}.get(int(b[2]))
    inside = b[0] + (1 << LOG2.get(int(b[2]), (0, 9))[1]) <= fp.mi_rows and b[1] + (1 << LOG2.get(int(b[2]), (9, 0))[0]) <= fp.mi_cols
    if b[3] or not kinds or not inside or room < 3 or rng.random() < (0.1 if b[2] == 9 else 0.4):
        return [b]
    parts = _split(b, *kinds[rng.integers(len(kinds))])
    room -= len(parts) - 1
    out = []
    for p in parts:
        cut = _cut(p, fp, rng, room)
        room -= len(cut) - 1
        out += cut
    return out


def cut_blocks(fp, blocks, sbs, seed):
    """The block lists with random intra blocks cut into smaller ones."""
    rng = np.random.default_rng(seed)
    blocks, sbs = blocks.copy(), sbs.copy()
    for s in range(fp.sb_cols * fp.sb_rows):
        first, n = sbs[s, :2]
        out, room = [], 64 - n
        for k in range(n):
            cut = _cut(blocks[first + k].copy(), fp, rng, room)
            room -= len(cut) - 1
            out += cut
        blocks[first:first + len(out)] = out
        sbs[s, 1] = len(out)
    return blocks, sbs


@pytest.mark.parametrize("turbo", [1, 0])
@pytest.mark.parametrize("w,h,seed", [(136, 104, 1), (200, 136, 2), (141, 99, 3), (352, 288, 4)])
def test_blocks_below_8x8(gpu, turbo, w, h, seed):
    print(f"\n[recon] blocks below 8x8, {w}x{h} turbo {turbo}", flush=True)
    cfg, fp, frames, blocks, sbs = _setup(w, h, "key", seed, turbo=turbo)
    blocks, sbs = cut_blocks(fp, blocks, sbs, seed)
    size = np.concatenate([blocks[f:f + n, 2] for f, n in sbs[:, :2]])
    assert np.isin(size, (0, 1, 2)).sum() > 20 and np.isin(size, (3, 6)).sum() > 20
    assert w < 352 or np.isin(size, (16, 17)).any()
    blocks, n_cfl, n_dir = libs.force_intra_modes(fp, blocks, sbs, seed)
    assert n_cfl > 0 and n_dir > 0
    _check(cfg, fp, frames, blocks, sbs)
