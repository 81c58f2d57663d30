/* The intra phase of the reconstruction on gfx950 (behaviour of
 * src/kernels/k_recon.h: recon_sb / recon_block / code_plane of intra
 * blocks, with the dependencies of src/backend_cpu.c:81-86): persistent
 * workgroups of 512 threads take superblocks in dependency order, with the
 * superblock's reconstruction, its surroundings and its source as LDS tiles.
 * Included by recon_intra.hip (frames without a luma search) and
 * recon_search.hip (transform type or depth search), which instantiate the
 * kernels: two smaller kernels instead of one with both paths, whose unused
 * path cost registers. Neither fits the 64 KB of instruction cache (about 300
 * and 550 KB, every stage inlined at each use). */
#ifndef MAV1_RECON_INTRA_H
#define MAV1_RECON_INTRA_H

#include "recon_lds.h"
#include "recon_queue.h"

#define TS_Y 132 /* tile row strides: 4 left columns + 128 (luma) / 64 (chroma) */
#define TS_C 68
#define TILE_Y (65 * TS_Y)
#define TILE_C (33 * TS_C)
#define TILE_BYTES (TILE_Y + 2 * TILE_C)

/* Per-wave LDS of the small intra blocks' prediction (edges, CfL). */
#define SI_EDGE (EDGE_NEG + 2 * 32 + 16)
struct SiWave {
  int eA[SI_EDGE], eL[SI_EDGE], ecp[2 * 32 + 40];
  int cfl[64], cflAvg, cflDc;
  long long aSse[33];
};

/* The depth search of a small intra block (tx_mode_select): luma blocks are
 * taken by teams of two waves, the deepest transform depth (4x4 transforms)
 * on one, the shallower depths on the other. Each wave reconstructs into a
 * private copy of the block with the samples its predictions read around it
 * (one row above, four columns left, twice the block's width and height). */
#define RD_TEAMS 3
#define RD_PS 52              /* row stride: 4 left columns + 2 * 16 samples, rounded up off a power of two */
#define RD_PIX (33 * RD_PS)
struct RdDeep {
  alignas(16) uint8_t pix[RD_PIX];
  alignas(16) int32_t lev[256];
};
struct RdShallow {
  SmallTx t;
  alignas(16) uint8_t pix[2][RD_PIX]; /* the depth being searched and the best one so far */
  alignas(16) int32_t lev[2][256];
};
/* What a depth's search found: cost, levels' types (a nibble per transform
 * block), transform blocks visited, any level, samples per transform block,
 * and the right / bottom end of the last block visited (CfL). */
struct RdRes {
  long long cost;
  unsigned long long types;
  int n, nz, area, depth, maxW, maxH, buf;
};

/* The working set of the workgroup that reconstructs a superblock's intra
 * blocks. */
struct RLds : RCommon {
  union {
    SmallTx sm[RW];
    BigTx big;
    int32_t cfl[32 * 32];
    struct {
      RdDeep deep[RD_TEAMS];
      RdShallow shal[RD_TEAMS];
      SmallTx ch[RW - 2 * RD_TEAMS];
    } rd;
  } u;
  long long aSse[33];
  int edgeA[EDGE_NEG + 2 * 64 + 32], edgeL[EDGE_NEG + 2 * 64 + 32], ecopy[2 * 64 + 40];
  uint8_t bd[3 * BDD * BDD];
  uint8_t bdSave[BDD * BDD];
  uint8_t save[64 * 64];
  /* the superblock's reconstruction with the row above it and four columns
   * left of it (luma row above: 128 samples wide, for the above-right edge),
   * and its source in the same layout */
  alignas(16) uint8_t tile[2][TILE_BYTES];
  /* the level schedule: the block records, per block the dependency level
   * (0: not a small intra block), the BlockDecoded bits its prediction reads
   * (above-right, below-left per plane) and the schedule (small intra blocks
   * by segment and level) */
  Mav1BlockInfo sbb[64];
  int plv[64], pav[64], pord[64];
  alignas(4) uint8_t cover[256]; /* per 4x4 cell of the superblock the index of its block */
  SiWave psw[RW];
  int ufl[64];              /* per block: U's CfL alpha is set (V's CfL waits for it) */
  int lerr;                 /* a wait ran out */
  /* per block the earlier intra blocks its prediction reads (bit j: block
   * j), and the blocks whose luma / U / V are done */
  unsigned long long dmask[64];
  unsigned long long ldm, udm, vdm;
  /* segments between the intra blocks the small-block path does not take:
   * per block the number of such blocks before it, the blocks themselves in
   * decode order, and per segment the end of its part of the schedule */
  int pseg[64], pbig[65], psegEnd[65], pnbig;
  /* the search: BlockDecoded bits around each block (bit k: the 4x4 cell k
   * right of the corner in the row above; bit 8 + k: k below it in the
   * column left), the end of its luma (CfL), each team's two results, how
   * many of them are there and the last block whose buffers are free */
  int pavl[64], pmaxW[64], pmaxH[64];
  RdRes rres[RD_TEAMS][2];
  int rjoin[RD_TEAMS], rrel[RD_TEAMS];
};
__shared__ RLds gL;

#include "recon_tx.h"

/* Pointer p into tile k (0: reconstruction, 1: source) of `plane` with
 * p[y * S + x] = sample (x, y) of the plane, for the superblock holding mi
 * (miRow, miCol); S = the tile's row stride. */
typedef __attribute__((address_space(3))) uint8_t lds_u8;
DEVI uint8_t *tile_ptr(int k, int plane, int miRow, int miCol, int &S) {
  const int sub = plane > 0;
  S = sub ? TS_C : TS_Y;
  lds_u8 *base = (lds_u8 *)(gL.tile[k] + (plane == 0 ? 0 : TILE_Y + (plane - 1) * TILE_C));
  const int oy = (((miRow >> 4) * 64) >> sub) - 1, ox = (((miCol >> 4) * 64) >> sub) - 4;
  /* the offset is taken off the 32-bit LDS address, so the pointer stays in
   * the LDS address space and its accesses are LDS instructions */
  return (uint8_t *)(lds_u8 *)(uintptr_t)((uint32_t)(uintptr_t)base - (uint32_t)(oy * S + ox));
}

/* Lane swaps within groups of 8 lanes. */
DEVI int lane_xor1(int v) { return dpp_t<DPP_QX1>(v); }
DEVI int lane_xor2(int v) { return dpp_t<DPP_QX2>(v); }
DEVI int lane_xor4(int v) { return dpp_t<DPP_HMIRROR>(dpp_t<0x1B>(v)); } /* 7 - i of 3 - i within the quad */
DEVI int lane_xor8(int v) { return dpp_t<DPP_MIRROR>(dpp_t<DPP_HMIRROR>(v)); } /* 15 - i of 7 - i within the half row */
/* a[j] of lane i <-> a[i] of lane j within each group of N lanes. */
template <int N>
DEVI void lane_transpose(int32_t (&a)[N], int r) {
#pragma unroll
  for (int b = 1; b < N; b <<= 1) {
    const bool hi = r & b;
#pragma unroll
    for (int i = 0; i < N; i++) {
      if (i & b) continue;
      const int32_t x0 = a[i], x1 = a[i | b], x = hi ? x0 : x1;
      const int32_t y = b == 1 ? lane_xor1(x) : b == 2 ? lane_xor2(x) : b == 4 ? lane_xor4(x) : lane_xor8(x);
      /* selects of values: a store to one of two elements would put the array in scratch memory */
      a[i] = hi ? y : x0;
      a[i | b] = hi ? x1 : y;
    }
  }
}
template <int N>
DEVI int lane_group_sum(int v) {
  v += lane_xor1(v);
  v += lane_xor2(v);
  if constexpr (N == 8) v += lane_xor4(v);
  return v;
}
template <int N>
DEVI int lane_group_max(int v) {
  v = d_max(v, lane_xor1(v));
  v = d_max(v, lane_xor2(v));
  if constexpr (N == 8) v = d_max(v, lane_xor4(v));
  return v;
}

/* Row, column and scan kind of a type (row_kind, col_kind, scan_kind), two
 * bits per type, for types that differ between lanes. */
constexpr uint32_t kind_table(int which) {
  const int row[16] = {0, 0, 1, 1, 0, 1, 1, 1, 1, 2, 2, 0, 2, 1, 2, 1};
  const int col[16] = {0, 1, 0, 1, 1, 0, 1, 1, 1, 2, 0, 2, 1, 2, 1, 2};
  const int scan[16] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1, 2, 1, 2, 1, 2};
  uint32_t v = 0;
  for (int t = 0; t < 16; t++) v |= (uint32_t)(which == 0 ? row[t] : which == 1 ? col[t] : scan[t]) << (2 * t);
  return v;
}

/* The inverse transform of a square block on lanes 0 .. N - 1 of a wave (and
 * alike on the other groups of N lanes): lane r enters with row r of the
 * dequantised coefficients in T and leaves with row r of the residual. */
template <int LN>
DEVI void lane_itx(int32_t (&T)[1 << LN], int rk, int ck, int r) {
  constexpr int N = 1 << LN, RS = LN - 2; /* Transform_Row_Shift of 4x4, 8x8, 16x16 */
  if (rk == 0) t_idct<LN>(T, 16);
  else if (rk == 1) t_1d<1, LN>(T, 16);
  else t_identity<LN>(T);
#pragma unroll
  for (int j = 0; j < N; j++) T[j] = d_clip(-(1 << 15), (1 << 15) - 1, d_round2(T[j], RS));
  lane_transpose<N>(T, r);
  if (ck == 0) t_idct<LN>(T, 16);
  else if (ck == 1) t_1d<1, LN>(T, 16);
  else t_identity<LN>(T);
  lane_transpose<N>(T, r);
#pragma unroll
  for (int j = 0; j < N; j++) T[j] = d_round2(T[j], 4);
}
typedef __attribute__((address_space(3))) uint32_t lds_u32;
/* One wave's reconstruction of a square block (tx_recon_small without a
 * flip): the levels q (LDS, stride N) dequantised, inverse transformed with
 * rows and columns changing place by lane swaps and added to px, whole words
 * at a time. Bound by the wave's serial chain: two LDS round trips fewer than
 * two passes over LDS with byte-wise adds, 2.4k cycles for a luma block of a
 * 1080p key frame instead of 3.1k. */
template <int LN>
DEVI void wave_recon(const int32_t *q_, int rk, int ck, int dcQ, int acQ, uint8_t *px, int S, int x, int y) {
  constexpr int N = 1 << LN;
  const int lane = d_local(threadIdx.x & 63), r = lane & (N - 1);
  const lds_i32 *q = lds(q_) + r * N;
  lds_u32 *pp = (lds_u32 *)(px + (y + r) * S + x);
  uint32_t pw[N / 4];
#pragma unroll
  for (int j = 0; j < N / 4; j++) pw[j] = pp[j];
  int32_t T[N];
#pragma unroll
  for (int j = 0; j < N; j++) {
    const int l = q[j], ad = __mul24(d_abs(l), (j == 0 && r == 0) ? dcQ : acQ) & 0xFFFFFF;
    T[j] = d_clip(-(1 << 15), (1 << 15) - 1, l < 0 ? -ad : ad);
  }
  lane_itx<LN>(T, rk, ck, r);
  uint32_t rw[N / 4];
#pragma unroll
  for (int j = 0; j < N / 4; j++) rw[j] = 0;
#pragma unroll
  for (int j = 0; j < N; j++) {
    const int sh = 8 * (j & 3);
    rw[j >> 2] |= (uint32_t)d_clip1((int)((pw[j >> 2] >> sh) & 255) + T[j]) << sh;
  }
  if (lane < N) {
#pragma unroll
    for (int j = 0; j < N / 4; j++) pp[j] = rw[j];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
/* tx_recon_small of an intra block (no flipped types). */
DEVI void wave_recon_any(const TxCtx &c, const int32_t *q, int32_t *res, int txSz, int type, int dcQ, int acQ,
                         uint8_t *px, int S, int x, int y) {
  txSz = d_uni(txSz);
  type = d_uni(type);
  const int rk = row_kind(type), ck = col_kind(type);
  if (txSz == TX_4X4) wave_recon<2>(q, rk, ck, dcQ, acQ, px, S, x, y);
  else if (txSz == TX_8X8) wave_recon<3>(q, rk, ck, dcQ, acQ, px, S, x, y);
  else if (txSz == TX_16X16) wave_recon<4>(q, rk, ck, dcQ, acQ, px, S, x, y);
  else tx_recon_small(c, q, res, SRS, txSz, type, dcQ, acQ, px, S, x, y);
}

/* The transform types of a 4x4 (LN 2) or 8x8 (LN 3) intra luma block side by
 * side on one wave: candidate type k of the list `types` (nc <= 8 nibbles,
 * none of them flipped) on lanes k * N .. k * N + N - 1, one lane per row or
 * column. A lane keeps its row or column in registers through the residual,
 * the two forward passes, the quantiser, the dequantiser and the two inverse
 * passes; rows and columns change place by lane swaps, so the search has no
 * LDS round trip besides its tables. Same values as tx_eval of each type,
 * then the first minimum: the levels go to lev (stride N), the
 * reconstruction into px (row stride S) at (x, y). Every lane of the wave
 * calls it; *type / *eob / the cost are the same in every lane.
 * Bound by one wave's issue rate (a serial chain): 8.6k cycles for an 8x8 and
 * 3.1k for a 4x4; the eight waves of tx_eval took 11.7k and 9.7k, with five
 * barriers around them, and this search with its passes through LDS 17k and
 * 7.9k. */
template <int LN>
DEVI long long wave_tx_search(const Mav1FrameParams &fp, const uint8_t *spx, int SS, uint8_t *px, int S, int x, int y,
                              unsigned long long types, int nc, int32_t *lev_, int *typeOut, int *eobOut) {
  constexpr int N = 1 << LN, SH = LN == 3 ? 5 : 4; /* Transform_Row_Shift + 4 */
  constexpr uint32_t RK = kind_table(0), CK = kind_table(1), SK = kind_table(2);
  const int lane = d_local(threadIdx.x & 63), r = lane & (N - 1), gi = lane >> LN;
  nc = d_uni(nc);
  const int t = (int)(types >> (4 * (gi < nc ? gi : 0))) & 15;
  const int rk = (RK >> (2 * t)) & 3, ck = (CK >> (2 * t)) & 3;
  const int dcQ = fp.dc_q[0], acQ = fp.ac_q[0], addDc = tx_quant_add(dcQ, true), addAc = tx_quant_add(acQ, false);
  const float rDc = gL.qrcp[0][0], rAc = gL.qrcp[0][1];
  /* row r of the source and the prediction */
  uint32_t sw[N / 4], pw[N / 4];
  const lds_u32 *sp = (const lds_u32 *)(spx + (y + r) * SS + x);
  lds_u32 *pp = (lds_u32 *)(px + (y + r) * S + x);
#pragma unroll
  for (int j = 0; j < N / 4; j++) {
    sw[j] = sp[j];
    pw[j] = pp[j];
  }
  const lds_i16 *is = (const lds_i16 *)(gL.iscans + ((SK >> (2 * t)) & 3) * SCAN_SMALL + (LN == 2 ? 0 : 16));
  int pos[N];
#pragma unroll
  for (int k = 0; k < N; k++) pos[k] = is[k * N + r];
  int32_t d[N];
#pragma unroll
  for (int j = 0; j < N; j++) d[j] = (int)((sw[j >> 2] >> (8 * (j & 3))) & 255) - (int)((pw[j >> 2] >> (8 * (j & 3))) & 255);
  /* forward rows, then columns (lane r holds column r) and the quantiser */
  const lds_i32 *Mh = lds(gL.smats) + rk * 336 + (LN == 2 ? 0 : 16), *Mv = lds(gL.smats) + ck * 336 + (LN == 2 ? 0 : 16);
  int32_t T[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    int s = 32768;
#pragma unroll
    for (int j = 0; j < N; j++) s += __mul24(d[j], Mh[k * N + j]);
    T[k] = s >> 16;
  }
  lane_transpose<N>(T, r);
  int32_t q[N];
  int eob = 0;
#pragma unroll
  for (int k = 0; k < N; k++) {
    long long s = 0;
#pragma unroll
    for (int i = 0; i < N; i++) s += (long long)Mv[k * N + i] * T[i];
    const bool dc = k == 0 && r == 0;
    q[k] = tx_quant_small(tx_round_col(s, SH), dc ? dcQ : acQ, dc ? addDc : addAc, dc ? rDc : rAc);
    eob = d_max(eob, q[k] ? pos[k] + 1 : 0);
  }
  eob = lane_group_max<N>(eob);
  /* the rate (tx_bits) and the dequantised levels */
  int bits = 0;
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int l = d_abs(q[k]);
    /* 8 (2 + 2 floor(log2 l)) = 16 (32 - clz(l)); 6 for a zero */
    const int lb = l ? 16 * (32 - __clz(l)) : 6;
    bits += pos[k] < eob ? lb : 0;
    const int ad = __mul24(l, (k == 0 && r == 0) ? dcQ : acQ) & 0xFFFFFF;
    T[k] = d_clip(-(1 << 15), (1 << 15) - 1, q[k] < 0 ? -ad : ad);
  }
  bits = lane_group_sum<N>(bits);
  bits = eob ? 48 + 16 * d_floorlog2((unsigned)eob + 1) + bits : 8;
  lane_transpose<N>(T, r);
  lane_itx<LN>(T, rk, ck, r);
  /* on rows: the reconstruction and its SSE */
  int e = 0;
  uint32_t rw[N / 4];
#pragma unroll
  for (int j = 0; j < N / 4; j++) rw[j] = 0;
#pragma unroll
  for (int j = 0; j < N; j++) {
    const int sh = 8 * (j & 3);
    const int v = d_clip1((int)((pw[j >> 2] >> sh) & 255) + T[j]);
    const int dd = (int)((sw[j >> 2] >> sh) & 255) - v;
    e += __mul24(dd, dd);
    rw[j >> 2] |= (uint32_t)v << sh;
  }
  e = lane_group_sum<N>(e);
  const long long cost = (long long)e * 16 + (long long)fp.lambda * bits / 8;
  /* the first minimum over the candidates: cost < 2^40, so the candidate
   * index fits beside it */
  long long best = LLONG_MAX;
  const long long key = gi < nc ? cost << 4 | gi : LLONG_MAX;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)key, k * N);
    const int hi = __builtin_amdgcn_readlane((int)(key >> 32), k * N);
    const long long c = (long long)(((unsigned long long)(unsigned)hi << 32) | lo);
    best = c < best ? c : best;
  }
  const int win = (int)best & 15;
  const int we = __builtin_amdgcn_readlane(eob, win * N);
  *typeOut = we > 0 ? (int)(types >> (4 * win)) & 15 : DCT_DCT;
  *eobOut = we;
  if (gi == win) {
    lds_i32 *lev = lds(lev_);
#pragma unroll
    for (int k = 0; k < N; k++) lev[k * N + r] = q[k];
#pragma unroll
    for (int j = 0; j < N / 4; j++) pp[j] = rw[j];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return best >> 4;
}

/* The single type of a 4x4 block on one wave (its four rows on the lanes of
 * each group of four): levels to lev, the reconstruction into px; returns
 * the eob. Same values as tx_eval and tx_recon_small. */
DEVI int wave_tx4(const Mav1FrameParams &fp, int plane, const uint8_t *spx, int SS, uint8_t *px, int S, int x, int y,
                  int t, int32_t *lev_) {
  const int lane = d_local(threadIdx.x & 63), r = lane & 3;
  const int rk = row_kind(t), ck = col_kind(t);
  const int dcQ = fp.dc_q[plane], acQ = fp.ac_q[plane];
  const float rDc = gL.qrcp[plane][0], rAc = gL.qrcp[plane][1];
  const uint32_t sw = *(const lds_u32 *)(spx + (y + r) * SS + x);
  lds_u32 *pp = (lds_u32 *)(px + (y + r) * S + x);
  const uint32_t pw = *pp;
  const lds_i32 *Mh = lds(gL.smats) + rk * 336, *Mv = lds(gL.smats) + ck * 336;
  int32_t d[4], T[4], q[4];
#pragma unroll
  for (int j = 0; j < 4; j++) d[j] = (int)((sw >> (8 * j)) & 255) - (int)((pw >> (8 * j)) & 255);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    int s = 32768;
#pragma unroll
    for (int j = 0; j < 4; j++) s += __mul24(d[j], Mh[k * 4 + j]);
    T[k] = s >> 16;
  }
  lane_transpose<4>(T, r);
  const lds_i16 *is = (const lds_i16 *)(gL.iscans + scan_kind(t) * SCAN_SMALL);
  int eob = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    long long s = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) s += (long long)Mv[k * 4 + i] * T[i];
    const bool dc = k == 0 && r == 0;
    q[k] = tx_quant_small(tx_round_col(s, 4), dc ? dcQ : acQ, dc ? tx_quant_add(dcQ, true) : tx_quant_add(acQ, false),
                          dc ? rDc : rAc);
    eob = d_max(eob, q[k] ? is[k * 4 + r] + 1 : 0);
  }
  eob = d_uni(lane_group_max<4>(eob));
  lds_i32 *lev = lds(lev_);
  if (lane < 4) {
#pragma unroll
    for (int k = 0; k < 4; k++) lev[k * 4 + r] = q[k];
  }
  if (eob > 0) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int ad = __mul24(d_abs(q[k]), (k == 0 && r == 0) ? dcQ : acQ) & 0xFFFFFF;
      T[k] = d_clip(-(1 << 15), (1 << 15) - 1, q[k] < 0 ? -ad : ad);
    }
    lane_transpose<4>(T, r);
    lane_itx<2>(T, rk, ck, r);
    uint32_t rw = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) rw |= (uint32_t)d_clip1((int)((pw >> (8 * j)) & 255) + T[j]) << (8 * j);
    if (lane < 4) *pp = rw;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  return eob;
}

/* ---- intra prediction of one transform block with the normative edge
 * preparation (7.11.2 incl. the edge filter and upsampling) ---- */
DEVI int edge_strength(int w, int h, int filterType, int delta) {
  int d = d_abs(delta), wh = w + h;
  if (filterType == 0) {
    if (wh <= 8) return d >= 56 ? 1 : 0;
    if (wh <= 16) return d >= 40 ? 1 : 0;
    if (wh <= 24) return d >= 32 ? 3 : d >= 16 ? 2 : d >= 8 ? 1 : 0;
    if (wh <= 32) return d >= 32 ? 3 : d >= 4 ? 2 : 1;
    return 3;
  }
  if (wh <= 8) return d >= 64 ? 2 : d >= 40 ? 1 : 0;
  if (wh <= 16) return d >= 48 ? 2 : d >= 20 ? 1 : 0;
  if (wh <= 24) return d >= 4 ? 3 : 0;
  return 3;
}
DEVI int use_upsample(int w, int h, int filterType, int delta) {
  int d = d_abs(delta);
  if (d <= 0 || d >= 40) return 0;
  return filterType == 0 ? (w + h <= 16) : (w + h <= 8);
}
/* 7.11.2.12 on e[-1 .. sz-2], by the team c with copy space cp */
DEVI void edge_filter(const TxCtx &c, int *e, int *cp, int sz, int strength) {
  if (!strength) return;
  for (int i = c.tid; i < sz; i += c.nt) cp[i] = e[i - 1];
  tx_sync(c);
  for (int i = 1 + c.tid; i < sz; i += c.nt) {
    int s = 0;
#pragma unroll
    for (int j = 0; j < 5; j++) s += INTRA_EDGE_KERNEL(strength - 1, j) * cp[d_clip(0, sz - 1, i - 2 + j)];
    e[i - 1] = (s + 8) >> 4;
  }
  tx_sync(c);
}
/* 7.11.2.11 */
DEVI void edge_upsample(const TxCtx &c, int *e, int *dup, int numPx) {
  for (int i = c.tid - 1; i < numPx; i += c.nt) dup[i + 2] = e[i];
  if (c.tid == 0) {
    dup[0] = e[-1];
    dup[numPx + 2] = e[numPx - 1];
  }
  tx_sync(c);
  if (c.tid == 0) e[-2] = dup[0];
  for (int i = c.tid; i < numPx; i += c.nt) {
    int s = -dup[i] + 9 * dup[i + 1] + 9 * dup[i + 2] - dup[i + 3];
    e[2 * i - 1] = d_clip1(d_round2(s, 4));
    e[2 * i] = dup[i + 2];
  }
  tx_sync(c);
}

/* Intra prediction of one transform block into px by the team c (the
 * workgroup or one wave), edge arrays eA / eL (addressed from -EDGE_NEG)
 * and copy space ecp. */
DEVI void intra_tx_predict(const TxCtx &c, uint8_t *px, int S, int sx, int sy, int lw, int lh, int mode, int delta,
                           int hl, int ha, int har, int hbl, int maxX, int maxY, int edgeFilter, int filterType,
                           int *eA, int *eL, int *ecp) {
  /* one transform block per team: the block's parameters are the same in
   * every lane */
  S = d_uni(S);
  sx = d_uni(sx);
  sy = d_uni(sy);
  lw = d_uni(lw);
  lh = d_uni(lh);
  mode = d_uni(mode);
  delta = d_uni(delta);
  hl = d_uni(hl);
  ha = d_uni(ha);
  har = d_uni(har);
  hbl = d_uni(hbl);
  filterType = d_uni(filterType);
  const int tid = c.tid, w = 1 << lw, h = 1 << lh;
  int *A = eA + EDGE_NEG, *Lc = eL + EDGE_NEG;
  /* 7.11.2 steps 1-3: the neighbouring samples */
  {
    const int aLim = d_min(maxX, sx + (har ? 2 * w : w) - 1), lLim = d_min(maxY, sy + (hbl ? 2 * h : h) - 1);
    for (int i = tid; i < w + h; i += c.nt) {
      A[i] = ha ? px[(sy - 1) * S + d_min(aLim, sx + i)] : hl ? px[sy * S + sx - 1] : 127;
      Lc[i] = hl ? px[d_min(lLim, sy + i) * S + sx - 1] : ha ? px[(sy - 1) * S + sx] : 129;
    }
    if (tid == 0) {
      const int corner = (ha && hl) ? px[(sy - 1) * S + sx - 1] : ha ? px[(sy - 1) * S + sx] : hl ? px[sy * S + sx - 1] : 128;
      A[-1] = Lc[-1] = corner;
    }
    tx_sync(c);
  }
  IntraMode im;
  intra_mode_setup(im, mode, delta, lw, lh);
  im.pAngle = d_uni(im.pAngle);
  im.dx = d_uni(im.dx);
  im.dy = d_uni(im.dy);
  im.corner = d_uni(A[-1]);
  if (mode >= V_PRED && mode <= D67_PRED && edgeFilter) {
    const int pa = im.pAngle;
    if (pa != 90 && pa != 180) {
      if (pa > 90 && pa < 180 && w + h >= 24) {
        const int v = d_round2(Lc[0] * 5 + A[-1] * 6 + A[0] * 5, 4);
        tx_sync(c);
        if (tid == 0) A[-1] = Lc[-1] = v;
        tx_sync(c);
      }
      if (ha)
        edge_filter(c, A, ecp, d_min(w, maxX - sx + 1) + (pa < 90 ? h : 0) + 1, edge_strength(w, h, filterType, pa - 90));
      if (hl)
        edge_filter(c, Lc, ecp, d_min(h, maxY - sy + 1) + (pa > 180 ? w : 0) + 1,
                    edge_strength(w, h, filterType, pa - 180));
    }
    im.upA = use_upsample(w, h, filterType, pa - 90);
    if (im.upA) edge_upsample(c, A, ecp, w + (pa < 90 ? h : 0));
    im.upL = use_upsample(w, h, filterType, pa - 180);
    if (im.upL) edge_upsample(c, Lc, ecp, h + (pa > 180 ? w : 0));
  }
  if (mode == DC_PRED) {
    long long s = 0;
    for (int i = tid; i < w; i += c.nt) s += ha ? A[i] : 0;
    for (int i = tid; i < h; i += c.nt) s += hl ? Lc[i] : 0;
    const int sum = (int)tx_sum64(c, s);
    im.dcv = (ha && hl) ? (sum + ((w + h) >> 1)) / (w + h) : hl ? d_clip1((sum + (h >> 1)) >> lh)
             : ha ? d_clip1((sum + (w >> 1)) >> lw) : 128;
  } else {
    im.dcv = 0;
  }
  for (int k = tid; k < w * h; k += c.nt) {
    const int i = k >> lw, j = k & (w - 1);
    px[(sy + i) * S + sx + j] = (uint8_t)intra_px(im, A, Lc, i, j);
  }
  tx_sync(c);
}

/* intra_tx_predict of a block of at most 8x8 by one wave: the edges stay in
 * registers, the row above on lanes 0 .. 31 (lane l: sample l - 1) and the
 * column left on lanes 32 .. 63, so that both are filtered and upsampled by
 * the same instructions, with lane permutes instead of copies through LDS.
 * Only the finished edges go to LDS (eA / eL), for the predictors that index
 * them. Same values; a luma block of a 1080p key frame 2.5k cycles instead of
 * 2.9k, a 4x4 of the depth search 2.2k instead of 3.0 - 4.4k. */
DEVI void wave_predict8(uint8_t *px, int S, int sx, int sy, int lw, int lh, int mode, int delta, int hl, int ha, int har,
                        int hbl, int maxX, int maxY, int edgeFilter, int filterType, int *eA, int *eL) {
  S = d_uni(S);
  sx = d_uni(sx);
  sy = d_uni(sy);
  lw = d_uni(lw);
  lh = d_uni(lh);
  mode = d_uni(mode);
  delta = d_uni(delta);
  hl = d_uni(hl);
  ha = d_uni(ha);
  har = d_uni(har);
  hbl = d_uni(hbl);
  const int lane = d_local(threadIdx.x & 63), half = lane >> 5, k = (lane & 31) - 1, w = 1 << lw, h = 1 << lh;
  const lds_u8 *lpx = (const lds_u8 *)px;
  /* 7.11.2 steps 1-3: the neighbouring samples */
  int e;
  if (ha || hl) {
    const int aLim = d_min(maxX, sx + (har ? 2 * w : w) - 1), lLim = d_min(maxY, sy + (hbl ? 2 * h : h) - 1);
    int X = half ? sx - 1 : d_min(aLim, sx + k), Y = half ? d_min(lLim, sy + k) : sy - 1;
    if (!(ha && hl)) {
      const bool mine = k >= 0 && (half ? hl : ha);
      if (!mine) {
        X = ha ? sx : sx - 1;
        Y = ha ? sy - 1 : sy;
      }
    }
    e = lpx[Y * S + X];
  } else {
    e = k < 0 ? 128 : half ? 129 : 127;
  }
  IntraMode im;
  intra_mode_setup(im, mode, delta, lw, lh);
  im.pAngle = d_uni(im.pAngle);
  im.dx = d_uni(im.dx);
  im.dy = d_uni(im.dy);
  im.corner = __builtin_amdgcn_readlane(e, 0);
  im.dcv = 0;
  if (mode == DC_PRED) {
    const bool use = k >= 0 && (half ? hl && k < h : ha && k < w);
    const int sum = wave_sum_dpp(use ? e : 0);
    im.dcv = (ha && hl) ? (lw == lh ? (sum + w) >> (lw + 1) : (sum + ((w + h) >> 1)) / (w + h))
             : hl       ? (sum + (h >> 1)) >> lh
             : ha       ? (sum + (w >> 1)) >> lw
                        : 128;
  } else {
    int up = 0; /* this half's edge is upsampled */
    int e2 = 0;
    if (mode >= V_PRED && mode <= D67_PRED && edgeFilter) {
      const int pa = im.pAngle;
      if (pa != 90 && pa != 180) {
        const int sA = ha ? edge_strength(w, h, filterType, pa - 90) : 0;
        const int sL = hl ? edge_strength(w, h, filterType, pa - 180) : 0;
        if (d_uni(sA | sL)) {
          const int st = half ? sL : sA;
          const int sz = half ? d_min(h, maxY - sy + 1) + (pa > 180 ? w : 0) + 1 : d_min(w, maxX - sx + 1) + (pa < 90 ? h : 0) + 1;
          const int i = k + 1, base = lane & 32;
          const int c0 = __shfl(e, base + d_clip(0, sz - 1, i - 2)), c1 = __shfl(e, base + d_clip(0, sz - 1, i - 1));
          const int c3 = __shfl(e, base + d_clip(0, sz - 1, i + 1)), c4 = __shfl(e, base + d_clip(0, sz - 1, i + 2));
          /* the kernels of 7.11.2.12: {0 4 8 4 0}, {0 5 6 5 0}, {2 4 4 4 2} */
          const int k1 = st == 2 ? 5 : 4, k2 = st == 1 ? 8 : st == 2 ? 6 : 4;
          int s = k2 * e + k1 * (c1 + c3);
          if (st == 3) s += 2 * (c0 + c4);
          if (st > 0 && i >= 1 && i < sz) e = (s + 8) >> 4;
        }
      }
      im.upA = d_uni(use_upsample(w, h, filterType, pa - 90));
      im.upL = d_uni(use_upsample(w, h, filterType, pa - 180));
      if (im.upA || im.upL) {
        up = half ? im.upL : im.upA;
        const int n = half ? h + (pa > 180 ? w : 0) : w + (pa < 90 ? h : 0), base = (lane & 32) + 1;
        const int m2 = __shfl(e, base + d_max(-1, k - 2)), m1 = __shfl(e, base + d_max(-1, k - 1));
        const int p1 = __shfl(e, base + d_min(n - 1, k + 1));
        e2 = d_clip1(d_round2(9 * (m1 + e) - m2 - p1, 4));
        /* lanes past the upsampled samples write nothing */
        if (up && k >= n) up = 2;
      }
    }
    lds_i32 *E = half ? lds(eL) + EDGE_NEG : lds(eA) + EDGE_NEG;
    if (up == 0) {
      if (k < w + h) E[k] = e;
    } else if (up == 1) {
      E[2 * k] = e;                  /* k = -1: the corner moves to -2 */
      if (k >= 0) E[2 * k - 1] = e2;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  if (lane < w * h) {
    const int i = lane >> lw, j = lane & (w - 1);
    px[(sy + i) * S + sx + j] = (uint8_t)intra_px(im, eA + EDGE_NEG, eL + EDGE_NEG, i, j);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
/* The prediction of a transform block by one wave. */
DEVI void wave_predict(uint8_t *px, int S, int sx, int sy, int lw, int lh, int mode, int delta, int hl, int ha, int har,
                       int hbl, int maxX, int maxY, int edgeFilter, int filterType, SiWave &W) {
  if (d_uni(lw) <= 3 && d_uni(lh) <= 3)
    wave_predict8(px, S, sx, sy, lw, lh, mode, delta, hl, ha, har, hbl, maxX, maxY, edgeFilter, filterType, W.eA, W.eL);
  else
    intra_tx_predict(wave_ctx(), px, S, sx, sy, lw, lh, mode, delta, hl, ha, har, hbl, maxX, maxY, edgeFilter,
                     filterType, W.eA, W.eL, W.ecp);
}

/* CfL (7.11.5) over the DC prediction in px: the alpha with the smallest
 * SSE against the source (first minimum over -16..16) unless given; the
 * alphas are scored one per wave. */
NOINL int cfl_tx(const uint8_t *luma, int LS, int sx, int sy, int maxLW, int maxLH, int lw, int lh, uint8_t *px, int S,
                 const uint8_t *__restrict__ spx, int alphaIn, int search, int excludeZero) {
  RLds &L = gL;
  const int tid = threadIdx.x, w = 1 << lw, h = 1 << lh, n = w * h;
  const int dcv = px[sy * S + sx]; /* DC prediction: one value over the block */
  long long s = 0;
  for (int k = tid; k < n; k += RT) {
    const int i = k >> lw, j = k & (w - 1);
    const int ly = d_min((sy + i) << 1, maxLH - 2), lx = d_min((sx + j) << 1, maxLW - 2);
    const uint8_t *l = luma + ly * LS + lx;
    const int v = ((int)l[0] + l[1] + l[LS] + l[LS + 1]) << 1;
    L.u.cfl[k] = v;
    s += v;
  }
  const int avg = d_round2((int)wg_sum64(s), lw + lh);
  int alpha = alphaIn;
  if (search) {
    const int wave = tid >> 6, lane = tid & 63;
    for (int a0 = -16; a0 <= 16; a0 += RW) {
      const int a = a0 + wave;
      if (a <= 16) {
        long long e = 0;
        for (int k = lane; k < n; k += 64) {
          const int i = k >> lw, j = k & (w - 1);
          const int d = d_clip1(dcv + d_round2signed(a * (L.u.cfl[k] - avg), 6)) - spx[(sy + i) * S + sx + j];
          e += d * d;
        }
        e = wave_sum64(e);
        if (lane == 0) L.aSse[a + 16] = e;
      }
    }
    __syncthreads();
    long long best = -1;
    for (int a = -16; a <= 16; a++) {
      if (a == 0 && excludeZero) continue;
      if (best < 0 || L.aSse[a + 16] < best) {
        best = L.aSse[a + 16];
        alpha = a;
      }
    }
  }
  for (int k = tid; k < n; k += RT) {
    const int i = k >> lw, j = k & (w - 1);
    px[(sy + i) * S + sx + j] = (uint8_t)d_clip1(dcv + d_round2signed(alpha * (L.u.cfl[k] - avg), 6));
  }
  __syncthreads();
  return alpha;
}

/* code_plane (k_recon.h:190-291) for the intra block in L.blk, in the
 * superblock's tiles, with the BlockDecoded flags; returns the cost. */
NOINL long long code_plane(const Mav1FrameParams &fp, int32_t *__restrict__ coefs, const int32_t *__restrict__ mats,
                           int plane, int txSz, int &maxLW, int &maxLH) {
  RLds &L = gL;
  Mav1BlockInfo &b = L.blk;
  const int tid = d_local(threadIdx.x);
  const int bs = b.bsize, sub = plane > 0;
  const int availU = b.mi_row > 0, availL = b.mi_col > tile_start(fp, b.mi_col);
  const int psz = SUBSAMPLED_SIZE(bs, sub, sub);
  const int n4w = Num_4x4_Blocks_Wide[psz], n4h = Num_4x4_Blocks_High[psz];
  const int baseX = (b.mi_col >> sub) * 4, baseY = (b.mi_row >> sub) * 4;
  int S, LS;
  uint8_t *px = tile_ptr(0, plane, b.mi_row, b.mi_col, S);
  const uint8_t *spx = tile_ptr(1, plane, b.mi_row, b.mi_col, S);
  const uint8_t *luma = tile_ptr(0, 0, b.mi_row, b.mi_col, LS);
  const int stepX = Tx_Width[txSz] >> 2, stepY = Tx_Height[txSz] >> 2;
  int cands[16], nc = 0;
  if (plane == 0) {
    const int set = get_tx_set(txSz, 0, fp.reduced_tx_set);
    if (!fp.tx_search || set == TX_SET_DCTONLY || fp.lossless) cands[nc++] = DCT_DCT;
    else
      for (int t = 0; t < 16; t++)
        if (in_set(set, t, 0)) cands[nc++] = t;
  } else {
    const int set = get_tx_set(txSz, 0, fp.reduced_tx_set);
    int t = Mode_To_Txfm[b.uv_mode];
    if (Tx_Size_Sqr_Up[txSz] > TX_32X32 || !in_set(set, t, 0)) t = DCT_DCT;
    cands[nc++] = t;
  }
  long long total = 0;
  int txIdx = 0, anyNz = 0;
  for (int y = 0; y < n4h; y += stepY)
    for (int x = 0; x < n4w; x += stepX) {
      const int sx = baseX + 4 * x, sy = baseY + 4 * y;
      if (sx >= ((fp.mi_cols * 4) >> sub) || sy >= ((fp.mi_rows * 4) >> sub)) continue;
      const int row = (sy << sub) >> 2, col = (sx << sub) >> 2, sbr = row & 15, sbc = col & 15;
      const int isCfl = plane > 0 && b.uv_mode == UV_CFL_PRED;
      const int lw = Tx_Width_Log2[txSz], lh = Tx_Height_Log2[txSz];
      intra_tx_predict(wg_ctx(), px, S, sx, sy, lw, lh, plane == 0 ? b.y_mode : (isCfl ? DC_PRED : b.uv_mode),
                       plane == 0 ? b.angle_y : b.angle_uv, availL || x > 0, availU || y > 0,
                       L.bd[BDI(plane, (sbr >> sub) - 1, (sbc >> sub) + stepX)],
                       L.bd[BDI(plane, (sbr >> sub) + stepY, (sbc >> sub) - 1)], ((fp.mi_cols * 4) >> sub) - 1,
                       ((fp.mi_rows * 4) >> sub) - 1, fp.enable_intra_edge_filter,
                       (b.interp_filter >> (plane == 0 ? 4 : 5)) & 1, L.edgeA, L.edgeL, L.ecopy);
      if (isCfl) {
        /* the first transform block searches the alpha, the others reuse it */
        const int search = txIdx == 0;
        const int a = cfl_tx(luma, LS, sx, sy, maxLW, maxLH, lw, lh, px, S, spx,
                             search ? 0 : plane == 1 ? b.cfl_alpha_u : b.cfl_alpha_v, search,
                             search && plane == 2 && b.cfl_alpha_u == 0);
        if (txIdx == 0 && tid == 0) {
          if (plane == 1) b.cfl_alpha_u = a;
          else b.cfl_alpha_v = a;
        }
        __syncthreads();
      }
      if (plane == 0) {
        maxLW = sx + stepX * 4;
        maxLH = sy + stepY * 4;
      }
      int t = DCT_DCT;
      long long c = 0;
      const int eob = code_tx_block(fp, spx, px, S, sx, sy, txSz, plane, cands, nc,
                                    coefs + b.coef_off[plane] + txIdx * Tx_Width[txSz] * Tx_Height[txSz], mats, &t,
                                    &c);
      total += c;
      if (plane == 0 && tid == 0) {
        if (txIdx < 16) {
          const int sh = 4 * (txIdx & 7);
          uint32_t *f = (uint32_t *)(txIdx < 8 ? &b.tx_types_lo : &b.tx_types_hi);
          *f = (*f & ~(15u << sh)) | ((uint32_t)t << sh);
        }
        if (txIdx == 0) b.tx_type = t;
      }
      anyNz |= eob > 0;
      txIdx++;
      if (tid == 0)
        for (int i = 0; i < stepY; i++)
          for (int j = 0; j < stepX; j++) L.bd[BDI(plane, (sbr >> sub) + i, (sbc >> sub) + j)] = 1;
      __syncthreads();
    }
  if (tid == 0) b.eob[plane] = anyNz;
  __syncthreads();
  return total;
}

/* recon_block (k_recon.h:293-394) for the intra block in L.blk, by the whole
 * workgroup. RD: with the luma depth search of tx_mode_select. */
template <bool RD>
NOINL void recon_intra_block(const Mav1FrameParams &fp, int32_t *__restrict__ coefs, const int32_t *__restrict__ mats) {
  RLds &L = gL;
  Mav1BlockInfo &b = L.blk;
  const int tid = threadIdx.x;
  const int bs = b.bsize;
  int maxLW = 0, maxLH = 0;
  if (tid == 0) {
    b.tx_depth = 0;
    b.interp_filter &= 0x30;
  }
  __syncthreads();
  for (int plane = 0; plane < 3; plane++) {
    /* transform size: 4x4 when lossless, the chroma size, or the luma size
     * of the best tx_depth */
    const int baseTx = fp.lossless ? TX_4X4 : plane > 0 ? uv_tx_size(bs) : Max_Tx_Size_Rect[bs];
    const int maxDepth = (RD && plane == 0 && !fp.lossless && fp.tx_mode_select) ? d_min(MAX_TX_DEPTH, Max_Tx_Depth[bs]) : 0;
    if (maxDepth == 0) {
      code_plane(fp, coefs, mats, plane, baseTx, maxLW, maxLH);
      continue;
    }
    if constexpr (RD) {
      const int w = BLOCK_WIDTH(bs), h = BLOCK_HEIGHT(bs);
      int TS;
      uint8_t *px = tile_ptr(0, 0, b.mi_row, b.mi_col, TS) + b.mi_row * 4 * TS_Y + b.mi_col * 4;
      for (int k = tid; k < w * h; k += RT) L.save[k] = px[(k / w) * TS_Y + (k % w)];
      for (int k = tid; k < BDD * BDD; k += RT) L.bdSave[k] = L.bd[k];
      __syncthreads();
      long long best = -1;
      int bestD = 0;
      for (int d = 0; d <= maxDepth + 1; d++) {
        const int depth = d <= maxDepth ? d : bestD;
        if (d == maxDepth + 1 && bestD == maxDepth) break;
        if (d > 0) {
          for (int k = tid; k < w * h; k += RT) px[(k / w) * TS_Y + (k % w)] = L.save[k];
          for (int k = tid; k < BDD * BDD; k += RT) L.bd[k] = L.bdSave[k];
          __syncthreads();
        }
        int t = baseTx;
        for (int k = 0; k < depth; k++) t = Split_Tx_Size[t];
        const long long c = code_plane(fp, coefs, mats, plane, t, maxLW, maxLH) +
                            (long long)fp.lambda * 8 * depth;
        if (d <= maxDepth && (best < 0 || c < best)) {
          best = c;
          bestD = depth;
        }
      }
      if (tid == 0) b.tx_depth = bestD;
      __syncthreads();
    }
  }
}

/* ---- small intra blocks ----
 * Intra blocks of 8x8 .. 16x16 have one transform block per plane (with a
 * depth search, of luma after the search's choice). */
DEVI bool si_small(const Mav1FrameParams &fp, const Mav1BlockInfo &b) {
  const int bs = b.bsize;
  return !b.is_inter && !fp.lossless &&
         (bs == BLOCK_8X8 || bs == BLOCK_8X16 || bs == BLOCK_16X8 || bs == BLOCK_16X16);
}

/* The BlockDecoded marks of one plane of block b, transform block by
 * transform block as code_plane sets them (one thread). */
DEVI void si_mark_g(const Mav1FrameParams &fp, int bs, int miRow, int miCol, int plane) {
  const int sub = plane > 0;
  const int txSz = fp.lossless ? TX_4X4 : plane ? uv_tx_size(bs) : Max_Tx_Size_Rect[bs];
  const int psz = SUBSAMPLED_SIZE(bs, sub, sub), n4w = Num_4x4_Blocks_Wide[psz], n4h = Num_4x4_Blocks_High[psz];
  const int baseX = (miCol >> sub) * 4, baseY = (miRow >> sub) * 4;
  const int stepX = Tx_Width[txSz] >> 2, stepY = Tx_Height[txSz] >> 2;
  for (int y = 0; y < n4h; y += stepY)
    for (int x = 0; x < n4w; x += stepX) {
      const int sx = baseX + 4 * x, sy = baseY + 4 * y;
      if (sx >= ((fp.mi_cols * 4) >> sub) || sy >= ((fp.mi_rows * 4) >> sub)) continue;
      const int sbr = ((sy << sub) >> 2) & 15, sbc = ((sx << sub) >> 2) & 15;
      for (int i = 0; i < stepY; i++)
        for (int j = 0; j < stepX; j++) gL.bd[BDI(plane, (sbr >> sub) + i, (sbc >> sub) + j)] = 1;
    }
}
DEVI void si_mark(const Mav1FrameParams &fp, const Mav1BlockInfo &b, int plane) {
  si_mark_g(fp, b.bsize, b.mi_row, b.mi_col, plane);
}

/* Geometry of plane `plane` of small block b. */
struct SiGeo {
  int sub, txSz, lw, lh, sx, sy, S;
  uint8_t *px;
  const uint8_t *spx;
};
DEVI SiGeo si_geo(const Mav1BlockInfo &b, int plane) {
  /* one block per wave: every field is the same in each lane */
  SiGeo g;
  plane = d_uni(plane);
  const int bs = d_uni(b.bsize), mr = d_uni(b.mi_row), mc = d_uni(b.mi_col);
  g.sub = plane > 0;
  g.txSz = d_uni(plane ? uv_tx_size(bs) : Max_Tx_Size_Rect[bs]);
  g.lw = d_uni(Tx_Width_Log2[g.txSz]);
  g.lh = d_uni(Tx_Height_Log2[g.txSz]);
  g.sx = (mc >> g.sub) * 4;
  g.sy = (mr >> g.sub) * 4;
  g.px = tile_ptr(0, plane, mr, mc, g.S);
  g.spx = tile_ptr(1, plane, mr, mc, g.S);
  return g;
}

/* Prediction of one plane of small block b by one wave (code_plane's
 * intra_tx_predict call) with its BlockDecoded bits above right (har) and
 * below left (hbl); for CfL also the alphas' SSEs (cfl_tx), with the end of
 * the coded luma (cflW, cflH; -1: the block's one transform block). */
DEVI void si_predict(const Mav1FrameParams &fp, Mav1BlockInfo &b, int plane, SiWave &W, int har, int hbl, int cflW = -1,
                     int cflH = -1) {
  const TxCtx c = wave_ctx();
  const int lane = c.tid;
  const SiGeo g = si_geo(b, plane);
  plane = d_uni(plane);
  const int sub = g.sub, mr = d_uni(b.mi_row), mc = d_uni(b.mi_col);
  const int availU = mr > 0, availL = mc > tile_start(fp, mc);
  const int uvMode = d_uni(b.uv_mode);
  const int isCfl = plane > 0 && uvMode == UV_CFL_PRED;
  wave_predict(g.px, g.S, g.sx, g.sy, g.lw, g.lh, d_uni(plane == 0 ? b.y_mode : (isCfl ? DC_PRED : uvMode)),
                   d_uni(plane == 0 ? b.angle_y : b.angle_uv), availL, availU, har, hbl,
                   ((fp.mi_cols * 4) >> sub) - 1, ((fp.mi_rows * 4) >> sub) - 1, fp.enable_intra_edge_filter,
                   d_uni((b.interp_filter >> (plane == 0 ? 4 : 5)) & 1), W);
  if (!isCfl) return;
  /* CfL (7.11.5) over the DC prediction: the luma average of each sample,
   * then one alpha per lane */
  const int w = 1 << g.lw, h = 1 << g.lh, n = w * h;
  int LS;
  const uint8_t *luma = tile_ptr(0, 0, mr, mc, LS);
  const int lumaTx = d_uni(Max_Tx_Size_Rect[d_uni(b.bsize)]);
  const int maxLW = cflW >= 0 ? cflW : mc * 4 + d_uni(Tx_Width[lumaTx]);
  const int maxLH = cflH >= 0 ? cflH : mr * 4 + d_uni(Tx_Height[lumaTx]);
  const int dcv = g.px[g.sy * g.S + g.sx];
  int sum = 0;
  for (int k = lane; k < n; k += 64) {
    const int i = k >> g.lw, j = k & (w - 1);
    const int ly = d_min((g.sy + i) << 1, maxLH - 2), lx = d_min((g.sx + j) << 1, maxLW - 2);
    const uint8_t *l = luma + ly * LS + lx;
    const int v = ((int)l[0] + l[1] + l[LS] + l[LS + 1]) << 1;
    W.cfl[k] = v;
    sum += v;
  }
  const int avg = d_round2(wave_sum_dpp(sum), g.lw + g.lh);
  tx_sync(c);
  if (lane < 33) {
    const int a = lane - 16;
    long long e = 0;
    for (int k = 0; k < n; k++) {
      const int i = k >> g.lw, j = k & (w - 1);
      const int d = d_clip1(dcv + d_round2signed(a * (W.cfl[k] - avg), 6)) - g.spx[(g.sy + i) * g.S + g.sx + j];
      e += d * d;
    }
    W.aSse[lane] = e;
  }
  if (lane == 0) {
    W.cflAvg = avg;
    W.cflDc = dcv;
  }
  tx_sync(c);
}

/* CfL: the alpha of smallest SSE (first in -16..16, 0 excluded when asked),
 * applied to the DC prediction. */
DEVI int si_cfl_apply(const Mav1BlockInfo &b, int plane, SiWave &W, int excludeZero) {
  const TxCtx c = wave_ctx();
  const int lane = c.tid;
  const SiGeo g = si_geo(b, plane);
  const int w = 1 << g.lw, n = w << g.lh;
  long long v = (lane < 33 && !(excludeZero && lane == 16)) ? W.aSse[lane] : LLONG_MAX;
  int idx = lane;
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const long long ov = __shfl_xor(v, m);
    const int oi = __shfl_xor(idx, m);
    if (ov < v || (ov == v && oi < idx)) {
      v = ov;
      idx = oi;
    }
  }
  const int alpha = d_uni(idx) - 16, avg = d_uni(W.cflAvg), dcv = d_uni(W.cflDc);
  tx_sync(c);
  for (int k = lane; k < n; k += 64) {
    const int i = k >> g.lw, j = k & (w - 1);
    g.px[(g.sy + i) * g.S + g.sx + j] = (uint8_t)d_clip1(dcv + d_round2signed(alpha * (W.cfl[k] - avg), 6));
  }
  tx_sync(c);
  return alpha;
}

/* The chroma plane of small block b by one wave: its single transform type
 * (code_plane), levels, reconstruction. */
DEVI void si_code_chroma(const Mav1FrameParams &fp, Mav1BlockInfo &b, int plane, int32_t *__restrict__ coefs,
                         const int32_t *__restrict__ mats, SmallTx &T) {
  const TxCtx c = wave_ctx();
  const SiGeo g = si_geo(b, plane);
  const int set = d_uni(get_tx_set(g.txSz, 0, fp.reduced_tx_set));
  int t = d_uni(Mode_To_Txfm[d_uni(b.uv_mode)]);
  if (d_uni(Tx_Size_Sqr_Up[g.txSz]) > TX_32X32 || !d_uni(in_set(set, t, 0))) t = DCT_DCT;
  const int tw = d_min(32, 1 << g.lw), th = d_min(32, 1 << g.lh);
  int32_t *co = coefs + d_uni(b.coef_off[plane]);
  int eob;
  if (g.txSz == TX_4X4) {
    eob = wave_tx4(fp, plane, g.spx, g.S, g.px, g.S, g.sx, g.sy, t, T.q);
  } else {
    long long cost;
    eob = tx_eval<true>(c, fp, g.spx, g.S, g.px, g.S, g.sx, g.sy, g.txSz, plane, t, true, T.resid, SRS, T.tmp, T.coef,
                        T.q, T.dq, SQS, mats, &cost);
    if (eob > 0)
      wave_recon_any(c, T.q, T.resid, g.txSz, t, fp.dc_q[plane], fp.ac_q[plane], g.px, g.S, g.sx, g.sy);
  }
  for (int k = c.tid; k < tw * th; k += 64) co[k] = T.q[k];
  if (c.tid == 0) b.eob[plane] = eob > 0;
}

/* Waits (thread 0) until *flag is set; false when maxSpin polls ran out. */
DEVI bool wait_flag(const int *flag, int maxSpin) {
  for (int it = 0; it < maxSpin; it++) {
    if (__hip_atomic_load(flag, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT)) return true;
    __builtin_amdgcn_s_sleep(4);
  }
  return false;
}

/* ---- the level schedule of a superblock ----
 * A superblock's small intra blocks (8x8 .. 16x16: one transform block per
 * plane, or with tx_mode_select a luma depth search) are coded by dependency
 * level instead of strictly one after another. A block's level is one more than the highest level of the
 * earlier (decode order) intra blocks of the superblock that its prediction
 * may read: those covering the column left of it down to twice its height,
 * the row above it right to twice its width, or the corner; blocks of one
 * level are therefore independent. The BlockDecoded flags its prediction
 * reads (above-right, below-left, per plane) are those of decode order: the
 * superblock's initial flags, or set where an earlier block of the
 * superblock covers the cell (the cover map: per 4x4 luma cell the index of
 * its block; a chroma cell counts as its top left luma cell: where blocks
 * below 8x8 share it, that is the first of them, and each of them codes and
 * marks the whole cell). Covering whole blocks equals marking their transform
 * blocks inside the frame, and a cell outside the frame never changes a
 * prediction (the edge fetch clamps to the frame).
 * The other intra blocks (larger than 16x16, 4:1, or below 8x8, which the
 * analysis never chooses) cut the superblock into segments: the small blocks
 * before one are finished, the whole workgroup codes it, and the schedule
 * goes on behind it; levels count within a segment only.
 * The blocks run as a dataflow over these dependencies (lvl_dataflow below);
 * the level pass records per block the mask of the earlier intra blocks it
 * reads (dmask). Without loss no block is small. */
/* Whether block i's BlockDecoded flag of plane p's 4x4 cell (y, x) of the
 * superblock is set when its turn comes in decode order. */
DEVI int lvl_decoded(int i, int p, int y, int x) {
  const int sub = p > 0;
  if (gL.bd[BDI(p, y, x)]) return 1;
  if (y < 0 || x < 0 || y >= (16 >> sub) || x >= (16 >> sub)) return 0;
  return gL.cover[((y << sub) << 4) + (x << sub)] < i;
}
DEVI void lvl_schedule(const Mav1FrameParams &fp, int n) {
  RLds &L = gL;
  const int tid = threadIdx.x;
  if (tid < 64) ((uint32_t *)L.cover)[tid] = 0xFFFFFFFFu;
  __syncthreads();
  if (tid < n) {
    const Mav1BlockInfo &b = L.sbb[tid];
    const int r0 = b.mi_row & 15, c0 = b.mi_col & 15;
    const int r1 = d_min(16, r0 + Num_4x4_Blocks_High[b.bsize]), c1 = d_min(16, c0 + Num_4x4_Blocks_Wide[b.bsize]);
    for (int r = r0; r < r1; r++)
      for (int c = c0; c < c1; c++) L.cover[r * 16 + c] = (uint8_t)tid;
  }
  __syncthreads();
  /* the BlockDecoded bits each small intra block's prediction reads */
  for (int q = tid; q < n * 6; q += RT) {
    const int i = q / 6, p = (q >> 1) % 3, f = q & 1, sub = p > 0;
    const Mav1BlockInfo &b = L.sbb[i];
    if (!si_small(fp, b)) continue;
    const int txSz = p ? uv_tx_size(b.bsize) : Max_Tx_Size_Rect[b.bsize];
    const int stepX = Tx_Width[txSz] >> 2, stepY = Tx_Height[txSz] >> 2;
    const int by = (b.mi_row & 15) >> sub, bx = (b.mi_col & 15) >> sub;
    if (lvl_decoded(i, p, f ? by + stepY : by - 1, f ? bx - 1 : bx + stepX)) atomicOr(&L.pav[i], 1 << (2 * p + f));
  }
  if (fp.tx_mode_select || fp.tx_search)
    for (int q = tid; q < n * 8; q += RT) {
      const int i = q >> 3, f = (q >> 2) & 1, k = (q & 3) + 1;
      const Mav1BlockInfo &b = L.sbb[i];
      if (!si_small(fp, b) || k > (f ? Num_4x4_Blocks_High[b.bsize] : Num_4x4_Blocks_Wide[b.bsize])) continue;
      const int by = b.mi_row & 15, bx = b.mi_col & 15;
      if (lvl_decoded(i, 0, f ? by + k : by - 1, f ? bx - 1 : bx + k)) atomicOr(&L.pavl[i], 1 << (8 * f + k));
    }
  /* levels, in decode order on wave 0 (lane j: block j as a dependency) */
  if (tid < 64) {
    const int j = tid;
    int myLv = 0, rj = 0, cj = 0, hj = 0, wj = 0, intraJ = 0, smallJ = 0;
    if (j < n) {
      const Mav1BlockInfo &o = L.sbb[j];
      rj = o.mi_row & 15;
      cj = o.mi_col & 15;
      hj = Num_4x4_Blocks_High[o.bsize];
      wj = Num_4x4_Blocks_Wide[o.bsize];
      intraJ = !o.is_inter;
      smallJ = si_small(fp, o);
    }
    const unsigned long long big = __ballot(intraJ && !smallJ);
    const int segJ = __popcll(big & ((1ull << j) - 1));
    L.pseg[j] = segJ;
    if (intraJ && !smallJ) L.pbig[segJ] = j;
    if (j == 0) L.pnbig = __popcll(big);
    unsigned long long todo = __ballot(smallJ);
    while (todo) {
      const int i = __ffsll((unsigned long long)todo) - 1;
      todo &= todo - 1;
      const Mav1BlockInfo &b = L.sbb[i];
      const int r = d_uni(b.mi_row) & 15, c = d_uni(b.mi_col) & 15, bs = d_uni(b.bsize);
      const int h = d_uni(Num_4x4_Blocks_High[bs]), w = d_uni(Num_4x4_Blocks_Wide[bs]);
      const int seg = __popcll(big & ((1ull << i) - 1));
      bool dep = false;
      if (j < i && intraJ) {
        const bool left = c - 1 >= cj && c - 1 < cj + wj && r - 1 < rj + hj && r + 2 * h > rj;
        const bool above = r - 1 >= rj && r - 1 < rj + hj && c - 1 < cj + wj && c + 2 * w > cj;
        dep = left || above;
      }
      const unsigned long long dm = __ballot(dep);
      const int m = wave_max_dpp(dep && segJ == seg ? myLv : 0);
      if (j == i) {
        myLv = m + 1;
        L.dmask[i] = dm;
      }
    }
    if (j < n) L.plv[j] = myLv;
  }
  __syncthreads();
  /* the schedule: small intra blocks by segment, level, then decode order */
  if (tid < n && L.plv[tid] > 0) {
    const int lv = L.plv[tid], sg = L.pseg[tid];
    int pos = 0;
    for (int k = 0; k < n; k++) {
      const int l = L.plv[k], s2 = L.pseg[k];
      pos += l > 0 && (s2 < sg || (s2 == sg && (l < lv || (l == lv && k < tid))));
    }
    L.pord[pos] = tid;
  }
  if (tid >= 64 && tid - 64 <= L.pnbig) {
    int cnt = 0;
    for (int k = 0; k < n; k++) cnt += L.plv[k] > 0 && L.pseg[k] <= tid - 64;
    L.psegEnd[tid - 64] = cnt;
  }
  __syncthreads();
}

/* ---- the level schedule as a dataflow ----
 * Luma of block i waits for the luma of the blocks in dmask[i] (those its
 * prediction reads); U (V) of block i waits for its own luma and the U (V)
 * of the blocks in dmask[i] (the chroma prediction reads the same neighbours
 * at half resolution); V's CfL waits for U's alpha. Without a search waves
 * 0 .. LVL_LW - 1 take the luma tasks in schedule order (task u on wave
 * u % LVL_LW), the other waves the chroma tasks (U then V per block): chroma
 * has two tasks per block and they take as long as a luma task, so chroma
 * gets the larger share (measured on the 1080p key frame: 2 luma waves
 * 13.4 ms, 3: 13.75 ms, 4: 14.2 ms). With a search the luma blocks go to
 * teams of two waves (rd_luma below). Every task waits only for tasks
 * earlier in its kind's order, and luma waits for no chroma, so the earliest
 * unfinished task can always run: every wait ends. Waits are still bounded
 * (a wait that runs out sets lerr). */
#define LVL_SPIN (1 << 20)
#define LVL_LW 2 /* waves for the luma tasks; the others take U and V */
DEVI unsigned long long lds_load64(const unsigned long long *p) {
  const unsigned long long v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  return ((unsigned long long)(unsigned)d_uni((int)(v >> 32)) << 32) | (unsigned)d_uni((int)(unsigned)v);
}
/* Waits until (*m & need) == need and bit `own` of *own (if own) is set. */
DEVI void lvl_wait(const unsigned long long *m, unsigned long long need, const unsigned long long *own, int i) {
  for (int it = 0; it < LVL_SPIN; it++) {
    if ((lds_load64(m) & need) == need && (!own || ((lds_load64(own) >> i) & 1))) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
      return;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  if ((threadIdx.x & 63) == 0) gL.lerr = 1;
}
DEVI void lvl_publish(unsigned long long *m, int i) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_or(m, 1ull << i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
/* ---- the luma depth search of a small intra block ----
 * recon_block's search (k_recon.h:341-378) over the transform depths of a
 * small block's luma: every depth starts from the same surroundings, so the
 * depths run side by side, each in a private copy of the block (RdDeep /
 * RdShallow); the cheapest (the shallowest on a tie) goes into the tile. The
 * deepest depth of every small block is 4x4.
 * Bound by the serial chain of prediction and search on the longer wave. For
 * a 16x16 block that is the shallower depths' one: 86k cycles for the types of
 * the 16x16 transform, one after the other, and about 11k for each 8x8 block,
 * 130k in all, against 85k for the sixteen 4x4 blocks; for an 8x8 block it is
 * the deepest depth's one, 21k against 11k. Coding each transform block by
 * the whole workgroup took about 30k cycles with its five barriers (11.3M per
 * superblock); two waves per block and one block per team let independent
 * blocks, depths and chroma run side by side: five full-RD frames of 1280x720
 * took 289 ms, with this split 80 ms, with the waves' transforms in registers
 * 62 ms. */

/* The private pixel copy addressed by plane position, for the block at luma
 * (x0, y0). */
DEVI uint8_t *rd_pix(uint8_t *pix, int x0, int y0) {
  lds_u8 *base = (lds_u8 *)pix;
  return (uint8_t *)(lds_u8 *)(uintptr_t)((uint32_t)(uintptr_t)base - (uint32_t)((y0 - 1) * RD_PS + x0 - 4));
}

/* One depth of block b by one wave: prediction and transform search of its
 * transform blocks in order, levels into lev one block after another,
 * reconstruction into pix. av: pavl of the block. */
template <bool DEEP>
DEVI RdRes rd_depth(const Mav1FrameParams &fp, const Mav1BlockInfo &b, int depth, int av, uint8_t *pix, int32_t *lev,
                    SiWave &P, SmallTx *W) {
  const TxCtx c = wave_ctx();
  const int lane = c.tid;
  const int bs = d_uni(b.bsize), mr = d_uni(b.mi_row), mc = d_uni(b.mi_col);
  const int x0 = mc * 4, y0 = mr * 4, n4w = d_uni(Num_4x4_Blocks_Wide[bs]), n4h = d_uni(Num_4x4_Blocks_High[bs]);
  int txSz = d_uni(Max_Tx_Size_Rect[bs]);
  for (int k = 0; k < depth; k++) txSz = d_uni(Split_Tx_Size[txSz]);
  const int lw = d_uni(Tx_Width_Log2[txSz]), lh = d_uni(Tx_Height_Log2[txSz]);
  const int stepX = 1 << (lw - 2), stepY = 1 << (lh - 2), area = 1 << (lw + lh);
  int TS;
  const uint8_t *tile = tile_ptr(0, 0, mr, mc, TS), *spx = tile_ptr(1, 0, mr, mc, TS);
  uint8_t *px = rd_pix(pix, x0, y0);
  /* the surroundings: rows -1 .. h - 1 from the corner to twice the width,
   * then the left column to twice the height (inside the tile; rows below
   * it are never read) */
  {
    const int nc = 2 * n4w + 1, h = n4h * 4, cx = lane & 15, bottom = (mr | 15) * 4 + 3;
    if (cx < nc)
      for (int rr = (lane >> 4) - 1; rr < h; rr += 4)
        *(lds_u32 *)(px + (y0 + rr) * RD_PS + x0 - 4 + 4 * cx) =
            *(const lds_u32 *)(tile + (y0 + rr) * TS_Y + x0 - 4 + 4 * cx);
    if (lane < h && y0 + h + lane <= bottom)
      *(lds_u32 *)(px + (y0 + h + lane) * RD_PS + x0 - 4) = *(const lds_u32 *)(tile + (y0 + h + lane) * TS_Y + x0 - 4);
    tx_sync(c);
  }
  const int set = d_uni(get_tx_set(txSz, 0, fp.reduced_tx_set));
  const bool search = fp.tx_search && set != TX_SET_DCTONLY;
  const unsigned long long types = search ? lds_load64(&gT.candList[set]) : (unsigned long long)DCT_DCT;
  const int nc = search ? d_uni(gT.candCnt[set]) : 1;
  const int availU = mr > 0, availL = mc > tile_start(fp, mc);
  const int mode = d_uni(b.y_mode), delta = d_uni(b.angle_y), ft = d_uni((b.interp_filter >> 4) & 1);
  const int maxX = fp.mi_cols * 4, maxY = fp.mi_rows * 4;
  RdRes R;
  R.cost = (long long)fp.lambda * 8 * depth;
  R.types = 0;
  R.n = R.nz = 0;
  R.area = area;
  R.depth = depth;
  R.maxW = R.maxH = R.buf = 0;
  for (int ty = 0; ty < n4h; ty += stepY)
    for (int tx = 0; tx < n4w; tx += stepX) {
      const int sx = x0 + 4 * tx, sy = y0 + 4 * ty;
      if (sx >= maxX || sy >= maxY) continue;
      /* above-right: from the row above the block, or inside it the
       * transform row before; below-left: from the column left of the block */
      const int har = ty == 0 ? (av >> (tx + stepX)) & 1 : tx + stepX < n4w;
      const int hbl = tx == 0 ? (av >> (8 + ty + stepY)) & 1 : 0;
      const int hl = availL || tx > 0, ha = availU || ty > 0;
      if constexpr (DEEP)
        wave_predict8(px, RD_PS, sx, sy, 2, 2, mode, delta, hl, ha, har, hbl, maxX - 1, maxY - 1,
                      fp.enable_intra_edge_filter, ft, P.eA, P.eL);
      else
        wave_predict(px, RD_PS, sx, sy, lw, lh, mode, delta, hl, ha, har, hbl, maxX - 1, maxY - 1,
                     fp.enable_intra_edge_filter, ft, P);
      int32_t *lv = lev + R.n * area;
      int t = DCT_DCT, eob = 0;
      long long cost;
      if constexpr (DEEP) {
        cost = wave_tx_search<2>(fp, spx, TS_Y, px, RD_PS, sx, sy, types, nc, lv, &t, &eob);
      } else if (txSz == TX_8X8) {
        cost = wave_tx_search<3>(fp, spx, TS_Y, px, RD_PS, sx, sy, types, nc, lv, &t, &eob);
      } else {
        cost = -1;
        for (int k = 0; k < nc; k++) {
          const int tk = (int)(types >> (4 * k)) & 15;
          long long ck;
          const int ek = tx_eval<true>(c, fp, spx, TS_Y, px, RD_PS, sx, sy, txSz, 0, tk, false, W->resid, SRS, W->tmp,
                                       W->coef, W->q, W->dq, SQS, nullptr, &ck);
          if (cost < 0 || ck < cost) {
            cost = ck;
            eob = ek;
            t = ek > 0 ? tk : DCT_DCT;
            for (int e = lane; e < area; e += 64) lv[e] = W->q[e];
            tx_sync(c);
          }
        }
        if (eob > 0)
          wave_recon_any(c, lv, W->resid, txSz, t, fp.dc_q[0], fp.ac_q[0], px, RD_PS, sx, sy);
      }
      R.cost += cost;
      if (R.n < 16) R.types |= (unsigned long long)t << (4 * R.n);
      R.nz |= eob > 0;
      R.n++;
      R.maxW = sx + stepX * 4;
      R.maxH = sy + stepY * 4;
    }
  return R;
}

/* A team's wave has its result of block i (slot 0: the deepest depth, 1: the
 * best shallower one) in its buffers; the second of the two to get here
 * chooses, puts the choice into the tile and publishes the block. alone: the
 * block has one depth, this wave's. */
DEVI void rd_join(const Mav1FrameParams &fp, int i, int team, int slot, const RdRes &R, bool alone,
                  int32_t *__restrict__ coefs) {
  RLds &L = gL;
  const TxCtx c = wave_ctx();
  const int lane = c.tid;
  if (lane == 0) L.rres[team][slot] = R;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  int first = 0;
  if (alone) {
    if (lane == 0) L.rres[team][0] = R;
  } else if (lane == 0) first = __hip_atomic_fetch_add(&L.rjoin[team], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0;
  first = d_uni(first);
  if (first) {
    /* the other wave chooses; this one's buffers are free once it has */
    int it = 0;
    while (d_uni(__hip_atomic_load(&L.rrel[team], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) != i && it < LVL_SPIN) {
      __builtin_amdgcn_s_sleep(1);
      it++;
    }
    if (it == LVL_SPIN && lane == 0) L.lerr = 1;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    return;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  const RdRes &D = L.rres[team][0], &H = L.rres[team][1];
  const bool deep = D.cost < H.cost;
  const RdRes &B = deep ? D : H;
  const int bufB = d_uni(B.buf);
  uint8_t *pix = deep ? L.u.rd.deep[team].pix : L.u.rd.shal[team].pix[bufB];
  const int32_t *lev = deep ? L.u.rd.deep[team].lev : L.u.rd.shal[team].lev[bufB];
  Mav1BlockInfo &b = L.sbb[i];
  const int bs = d_uni(b.bsize), mr = d_uni(b.mi_row), mc = d_uni(b.mi_col), x0 = mc * 4, y0 = mr * 4;
  const int lw4 = d_uni(Num_4x4_Blocks_Wide[bs]) == 4 ? 2 : 1, n4h = d_uni(Num_4x4_Blocks_High[bs]);
  {
    int TS;
    uint8_t *tile = tile_ptr(0, 0, mr, mc, TS);
    const uint8_t *px = rd_pix(pix, x0, y0);
    const int rr = lane >> lw4, cc = (lane & ((1 << lw4) - 1)) * 4;
    if (rr < n4h * 4)
      *(lds_u32 *)(tile + (y0 + rr) * TS_Y + x0 + cc) = *(const lds_u32 *)(px + (y0 + rr) * RD_PS + x0 + cc);
  }
  if (lane == 0) {
    L.pmaxW[i] = B.maxW;
    L.pmaxH[i] = B.maxH;
    L.rjoin[team] = 0;
  }
  lvl_publish(&L.ldm, i);
  /* the levels of the chosen depth out, the block's transform fields */
  const int n = d_uni(B.n), cov = n * d_uni(B.area), nD = d_uni(D.n);
  int32_t *co = coefs + d_uni(b.coef_off[0]);
  for (int k = lane; k < cov; k += 64) co[k] = lev[k];
  if (lane == 0) {
    /* a type nibble that the choice does not set keeps what the deepest
     * depth, searched last, left there */
    const unsigned long long mB = n >= 16 ? ~0ull : (1ull << (4 * n)) - 1, mD = nD >= 16 ? ~0ull : (1ull << (4 * nD)) - 1;
    unsigned long long f = (unsigned long long)(uint32_t)b.tx_types_hi << 32 | (uint32_t)b.tx_types_lo;
    f = (f & ~mD) | (D.types & mD);
    f = (f & ~mB) | (B.types & mB);
    b.tx_types_lo = (int32_t)(uint32_t)f;
    b.tx_types_hi = (int32_t)(uint32_t)(f >> 32);
    b.tx_type = (int32_t)(B.types & 15);
    b.tx_depth = B.depth;
    b.eob[0] = B.nz;
    b.interp_filter &= 0x30;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if (lane == 0) __hip_atomic_store(&L.rrel[team], i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

/* One team wave's part of block i: the deepest depth (slot 0) or the others
 * (slot 1, the first minimum kept in one of two buffers). */
DEVI void rd_luma(const Mav1FrameParams &fp, int i, int team, int slot, int32_t *__restrict__ coefs, SiWave &P) {
  RLds &L = gL;
  const Mav1BlockInfo &b = L.sbb[i];
  const int av = d_uni(L.pavl[i]);
  const int maxD = fp.tx_mode_select ? d_min(MAX_TX_DEPTH, d_uni(Max_Tx_Depth[d_uni(b.bsize)])) : 0;
  RdRes R;
  if (slot == 0) {
    if (maxD == 0) return;
    RdDeep &W = L.u.rd.deep[team];
    R = rd_depth<true>(fp, b, maxD, av, W.pix, W.lev, P, nullptr);
  } else {
    RdShallow &W = L.u.rd.shal[team];
    int buf = 0;
    for (int d = 0; d < d_max(1, maxD); d++) {
      RdRes Q = rd_depth<false>(fp, b, d, av, W.pix[buf], W.lev[buf], P, &W.t);
      Q.buf = buf;
      if (d == 0) {
        /* depth 0 covers the block also outside the frame, where no deeper
         * depth writes: its levels stay there whatever is chosen */
        const int vw = d_min(fp.mi_cols - d_uni(b.mi_col), d_uni(Num_4x4_Blocks_Wide[d_uni(b.bsize)]));
        const int vh = d_min(fp.mi_rows - d_uni(b.mi_row), d_uni(Num_4x4_Blocks_High[d_uni(b.bsize)]));
        int32_t *co = coefs + d_uni(b.coef_off[0]);
        for (int k = vw * vh * 16 + (threadIdx.x & 63); k < Q.area; k += 64) co[k] = W.lev[buf][k];
      }
      if (d == 0 || Q.cost < R.cost) {
        R = Q;
        buf ^= 1;
      }
    }
  }
  rd_join(fp, i, team, slot, R, maxD == 0, coefs);
}

/* RD: the blocks' luma through the depth search (tx_mode_select). Blocks
 * pord[u0 .. u1). Teams take the luma blocks in schedule order (block u on
 * team u % RD_TEAMS), so a wave still waits only for blocks earlier in that
 * order. */
template <bool RD>
DEVI void lvl_dataflow(const Mav1FrameParams &fp, int32_t *__restrict__ coefs, const int32_t *__restrict__ mats, int u0,
                       int u1) {
  RLds &L = gL;
  const int wave = d_uni(threadIdx.x >> 6), lane = threadIdx.x & 63;
  constexpr int LW = RD ? 2 * RD_TEAMS : LVL_LW;
  u0 = d_uni(u0);
  u1 = d_uni(u1);
  const TxCtx c = wave_ctx();
  SiWave &P = L.psw[wave];
  if (wave < LW) {
    if constexpr (RD) {
      const int slot = wave < RD_TEAMS ? 0 : 1, team = wave - slot * RD_TEAMS;
      for (int u = u0 + team; u < u1; u += RD_TEAMS) {
        const int i = d_uni(L.pord[u]);
        lvl_wait(&L.ldm, L.dmask[i], nullptr, 0);
        rd_luma(fp, i, team, slot, coefs, P);
      }
    } else {
      SmallTx &W = L.u.sm[wave];
      for (int u = u0 + wave; u < u1; u += LVL_LW) {
        const int i = d_uni(L.pord[u]);
        Mav1BlockInfo &b = L.sbb[i];
        lvl_wait(&L.ldm, L.dmask[i], nullptr, 0);
        if (lane == 0) {
          b.tx_depth = 0;
          b.interp_filter &= 0x30;
        }
        const int av = d_uni(L.pav[i]);
        si_predict(fp, b, 0, P, av & 1, (av >> 1) & 1);
        const SiGeo g = si_geo(b, 0);
        long long cost;
        const int eob = tx_eval<true>(c, fp, g.spx, g.S, g.px, g.S, g.sx, g.sy, g.txSz, 0, DCT_DCT, true, W.resid, SRS,
                                      W.tmp, W.coef, W.q, W.dq, SQS, mats, &cost);
        /* the reconstruction first: the blocks waiting for this one read only
         * its pixels; then the levels out and the block's transform fields */
        if (eob > 0)
          wave_recon_any(c, W.q, W.resid, g.txSz, DCT_DCT, fp.dc_q[0], fp.ac_q[0], g.px, g.S, g.sx, g.sy);
        lvl_publish(&L.ldm, i);
        const int tw = d_min(32, 1 << g.lw), th = d_min(32, 1 << g.lh);
        int32_t *co = coefs + d_uni(b.coef_off[0]);
        for (int k = c.tid; k < tw * th; k += 64) co[k] = W.q[k];
        if (lane == 0) {
          b.tx_types_lo = (int32_t)(((uint32_t)b.tx_types_lo & ~15u) | (uint32_t)DCT_DCT);
          b.tx_type = DCT_DCT;
          b.eob[0] = eob > 0;
        }
      }
    }
  } else {
    SmallTx &W = RD ? L.u.rd.ch[wave - LW] : L.u.sm[wave];
    for (int ci = 2 * u0 + wave - LW; ci < 2 * u1; ci += RW - LW) {
      const int u = ci >> 1, plane = 1 + (ci & 1), i = d_uni(L.pord[u]);
      Mav1BlockInfo &b = L.sbb[i];
      unsigned long long *dn = plane == 1 ? &L.udm : &L.vdm;
      lvl_wait(dn, L.dmask[i], &L.ldm, i);
      const int av = d_uni(L.pav[i]);
      si_predict(fp, b, plane, P, (av >> (2 * plane)) & 1, (av >> (2 * plane + 1)) & 1, RD ? d_uni(L.pmaxW[i]) : -1,
                 RD ? d_uni(L.pmaxH[i]) : -1);
      if (d_uni(b.uv_mode) == UV_CFL_PRED) {
        if (plane == 1) {
          const int a = si_cfl_apply(b, 1, P, 0);
          if (lane == 0) {
            b.cfl_alpha_u = a;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __hip_atomic_store(&L.ufl[i], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        } else {
          int spin = 0;
          while (!d_uni(__hip_atomic_load(&L.ufl[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) &&
                 spin < LVL_SPIN) {
            __builtin_amdgcn_s_sleep(1);
            spin++;
          }
          if (spin == LVL_SPIN && lane == 0) L.lerr = 1;
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
          const int a = si_cfl_apply(b, 2, P, d_uni(b.cfl_alpha_u) == 0);
          if (lane == 0) b.cfl_alpha_v = a;
        }
      }
      si_code_chroma(fp, b, plane, coefs, mats, W);
      lvl_publish(dn, i);
    }
  }
  __syncthreads();
}

/* The intra blocks of superblock (r, c) (recon_sb, k_recon.h:396-440) in
 * two parts. intra_sb_prep: what does not read the neighbours'
 * reconstruction (BlockDecoded flags, source tile, block records, the level
 * schedule), so it can run while the neighbours are still being coded. */
DEVI void intra_sb_prep(const Mav1FrameParams &fp, const Mav1BlockInfo *__restrict__ blocks, const Mav1SbInfo &S,
                        const uint8_t *__restrict__ src, int r, int c) {
  RLds &L = gL;
  /* opaque, as in code_plane: addresses derived from it are not kept in
   * registers through the coding of the blocks (spilled VGPRs 31 -> 22, with a
   * search 53 -> 40; intra phase of a full-RD 1280x720 key frame 23.05 ->
   * 22.76 ms) */
  const int tid = d_local(threadIdx.x);
  /* clear_block_decoded_flags (k_recon.h:402-414) */
  const int mr = r * 16, mc = c * 16;
  const int tileEnd = d_min(fp.mi_cols, tile_start(fp, mc) + fp.tile_w_sb * 16);
  for (int q = tid; q < 3 * BDD * BDD; q += RT) {
    const int p = q / (BDD * BDD), e = q - p * BDD * BDD, y = e / BDD - 1, x = e % BDD - 1, sub = p > 0;
    const int w4 = (tileEnd - mc) >> sub, h4 = (fp.mi_rows - mr) >> sub;
    uint8_t v = (y < 0 && x < w4) ? 1 : (x < 0 && y < h4) ? 1 : 0;
    if (y == (16 >> sub) && x == -1) v = 0;
    if (y <= (16 >> sub) && x <= (16 >> sub)) L.bd[q] = v;
  }
  /* the superblock's source tile, as dwords */
  for (int p = 0; p < 3; p++) {
    const int sub = p > 0, TS = sub ? TS_C : TS_Y, n = 64 >> sub, wpr = TS / 4;
    const int oy = ((r * 64) >> sub) - 1, ox = ((c * 64) >> sub) - 4, stride = fp.stride[p];
    uint32_t *ts = (uint32_t *)(L.tile[1] + (p == 0 ? 0 : TILE_Y + (p - 1) * TILE_C));
    for (int q = tid; q < (n + 1) * wpr; q += RT) {
      const int ty = q / wpr, tx = (q - ty * wpr) * 4, Y = oy + ty, X = ox + tx;
      if (ty == 0 || tx < 4 || tx >= 4 + n || Y < 0 || X < 0 || X >= stride) continue;
      ts[q] = *(const uint32_t *)(src + fp.offset[p] + Y * stride + X);
    }
  }
  /* the block records */
  const int nb = S.num_blocks;
  for (int q = tid; q < nb * 27; q += RT) ((int32_t *)L.sbb)[q] = ((const int32_t *)(blocks + S.first_block))[q];
  for (int q = tid; q < 64; q += RT) {
    L.pav[q] = 0;
    L.pavl[q] = 0;
    L.ufl[q] = 0;
  }
  if (tid < RD_TEAMS) {
    L.rjoin[tid] = 0;
    L.rrel[tid] = -1;
  }
  if (tid == 0) {
    L.lerr = 0;
    L.ldm = L.udm = L.vdm = 0;
  }
  __syncthreads();
  lvl_schedule(fp, nb);
}

/* intra_sb: after intra_sb_prep and once the neighbouring superblocks are
 * done, the reconstruction tile (with the row above and the columns left),
 * the blocks, the tiles back. Returns non-zero when a wait inside ran out
 * (the results are then not to be used). */
/* RD: the frame searches transform types or depths. */
template <bool RD>
DEVI int intra_sb(const Mav1FrameParams &fp, Mav1BlockInfo *__restrict__ blocks, const Mav1SbInfo &S,
                  uint8_t *rec, int32_t *__restrict__ coefs, const int32_t *__restrict__ mats, int r, int c) {
  RLds &L = gL;
  const int tid = threadIdx.x;
  for (int p = 0; p < 3; p++) {
    const int sub = p > 0, TS = sub ? TS_C : TS_Y, n = 64 >> sub, wpr = TS / 4;
    const int oy = ((r * 64) >> sub) - 1, ox = ((c * 64) >> sub) - 4, stride = fp.stride[p];
    uint32_t *tr = (uint32_t *)(L.tile[0] + (p == 0 ? 0 : TILE_Y + (p - 1) * TILE_C));
    for (int q = tid; q < (n + 1) * wpr; q += RT) {
      const int ty = q / wpr, tx = (q - ty * wpr) * 4, Y = oy + ty, X = ox + tx;
      if ((ty > 0 && tx >= 4 + n) || Y < 0 || X < 0 || X >= stride) continue;
      tr[q] = *(const uint32_t *)(rec + fp.offset[p] + Y * stride + X);
    }
  }
  const int nb = S.num_blocks;
  __syncthreads();
  /* the segments of small blocks with the larger blocks between them */
  const int nbig = d_uni(L.pnbig);
  int u0 = 0, marked = 0;
  for (int sg = 0; sg <= nbig; sg++) {
    const int u1 = d_uni(L.psegEnd[sg]);
    if (u1 > u0) lvl_dataflow<RD>(fp, coefs, mats, u0, u1);
    u0 = u1;
    if (sg == nbig) break;
    /* a larger intra block: the flags of the blocks before it, then the
     * whole workgroup codes it */
    const int i = d_uni(L.pbig[sg]);
    for (int q = marked * 3 + tid; q < i * 3; q += RT) si_mark(fp, L.sbb[q / 3], q % 3);
    if (tid < 27) ((int32_t *)&L.blk)[tid] = ((const int32_t *)&L.sbb[i])[tid];
    __syncthreads();
    recon_intra_block<RD>(fp, coefs, mats);
    if (tid < 27) ((int32_t *)&L.sbb[i])[tid] = ((const int32_t *)&L.blk)[tid];
    if (tid == 0) {
      L.ldm |= 1ull << i;
      L.udm |= 1ull << i;
      L.vdm |= 1ull << i;
    }
    marked = i + 1;
    __syncthreads();
  }
  for (int q = tid; q < nb * 27; q += RT)
    if (!L.sbb[q / 27].is_inter) ((int32_t *)(blocks + S.first_block))[q] = ((const int32_t *)L.sbb)[q];
  __syncthreads();
  /* the superblock back into the frame */
  for (int p = 0; p < 3; p++) {
    const int sub = p > 0, TS = sub ? TS_C : TS_Y, n = 64 >> sub, wpr = n / 4;
    const int y0 = (r * 64) >> sub, x0 = (c * 64) >> sub, stride = fp.stride[p];
    const uint32_t *tr = (const uint32_t *)(L.tile[0] + (p == 0 ? 0 : TILE_Y + (p - 1) * TILE_C));
    for (int q = tid; q < n * wpr; q += RT) {
      const int ty = q / wpr, tx = (q - ty * wpr) * 4;
      *(uint32_t *)(rec + fp.offset[p] + (y0 + ty) * stride + x0 + tx) = tr[(ty + 1) * (TS / 4) + 1 + tx / 4];
    }
  }
  return L.lerr;
}
template <bool RD>
__global__ __launch_bounds__(RT) void k_recon_intra(const Mav1FrameParams fp, Mav1BlockInfo *__restrict__ blocks,
                                                    const Mav1SbInfo *__restrict__ sbs, const uint8_t *__restrict__ src,
                                                    uint8_t *rec, int32_t *__restrict__ coefs,
                                                    const int32_t *__restrict__ mats, int *__restrict__ iwork,
                                                    int maxSpin) {
  RLds &L = gL;
  const int tid = threadIdx.x, n = fp.sb_cols * fp.sb_rows;
  const int *list = iwork + IW_HDR, *has = list + n;
  int *done = iwork + IW_HDR + 2 * n;
  /* the first superblock before anything else: workgroups without one leave
   * at once */
  if (tid == 0) L.ival[2] = atomicAdd(&iwork[IW_NEXT], 1);
  __syncthreads();
  if (L.ival[2] >= iwork[IW_COUNT]) return;
  stage_tabs(tid, RT);
  stage_smats(fp, mats);
  for (;;) {
    const int idx = L.ival[2];
    __syncthreads();
    if (idx >= iwork[IW_COUNT]) break;
    const int sb = list[idx], r = sb / fp.sb_cols, c = sb - r * fp.sb_cols;
    /* everything that does not read the neighbours' reconstruction first,
     * beside the wait for them */
    intra_sb_prep(fp, blocks, sbs[sb], src, r, c);
    if (tid == 0) {
      /* the neighbours whose reconstruction this superblock reads */
      const int ts = (c / fp.tile_w_sb) * fp.tile_w_sb, te = d_min(fp.sb_cols, ts + fp.tile_w_sb);
      const int dep[4] = {c > ts ? sb - 1 : -1, r > 0 && c > ts ? sb - fp.sb_cols - 1 : -1, r > 0 ? sb - fp.sb_cols : -1,
                          r > 0 && c + 1 < te ? sb - fp.sb_cols + 1 : -1};
      for (int k = 0; k < 4; k++)
        if (dep[k] >= 0 && has[dep[k]] && !wait_flag(&done[dep[k]], maxSpin)) atomicOr(&iwork[IW_ERR], 1);
    }
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    const int err = intra_sb<RD>(fp, blocks, sbs[sb], rec, coefs, mats, r, c);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if (tid == 0) {
      if (err) atomicOr(&iwork[IW_ERR], 1);
      __hip_atomic_store(&done[sb], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      L.ival[2] = atomicAdd(&iwork[IW_NEXT], 1);
    }
    __syncthreads();
  }
}

template <bool RD>
__global__ __launch_bounds__(RT) void k_recon_intra_b(const BatchFrame *__restrict__ T, int nfr, int *__restrict__ q,
                                                      int maxSpin) {
  RLds &L = gL;
  const int tid = threadIdx.x;
  int staged = -1;
  for (;;) {
    if (tid == 0) {
      int v = -1;
      const int idx = atomicAdd(&q[QH_HEAD], 1);
      if (idx < q[QH_TOTAL]) {
        for (int it = 0; it < maxSpin && v < 0; it++) {
          v = __hip_atomic_load(&q[QH_ITEMS + idx], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
          if (v < 0) __builtin_amdgcn_s_sleep(4);
        }
        if (v < 0)
          for (int f = 0; f < nfr; f++) atomicOr(&T[f].iwork[IW_ERR], 1);
      }
      L.ival[2] = v;
    }
    __syncthreads();
    const int v = L.ival[2];
    __syncthreads();
    if (v < 0) break;
    const int f = v >> 16, sb = v & 0xffff;
    const BatchFrame &F = T[f];
    const Mav1FrameParams &fp = F.fp;
    if (staged < 0) stage_tabs(tid, RT);
    if (staged != f) {
      stage_smats(fp, gptr(F.mats));
      staged = f;
    }
    __syncthreads();
    const int r = sb / fp.sb_cols, c = sb - r * fp.sb_cols;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    intra_sb_prep(fp, gptr(F.blocks), gptr(F.sbs)[sb], gptr(F.src), r, c);
    const int err = intra_sb<RD>(fp, gptr(F.blocks), gptr(F.sbs)[sb], gptr(F.rec), gptr(F.coefs), gptr(F.mats), r, c);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if (tid == 0) {
      if (err) atomicOr(&gptr(F.iwork)[IW_ERR], 1);
      /* the superblocks that read this one: queued when this was their last
       * pending dependency */
      const int n = fp.sb_cols * fp.sb_rows;
      const int *has = gptr(F.iwork) + IW_HDR + n;
      int *cnt = gptr(F.iwork) + IW_HDR + 3 * n;
      const int cand[4] = {c + 1 < fp.sb_cols ? sb + 1 : -1, r + 1 < fp.sb_rows && c + 1 < fp.sb_cols ? sb + fp.sb_cols + 1 : -1,
                           r + 1 < fp.sb_rows ? sb + fp.sb_cols : -1, r + 1 < fp.sb_rows && c > 0 ? sb + fp.sb_cols - 1 : -1};
      for (int k = 0; k < 4; k++) {
        const int d = cand[k];
        if (d < 0 || !has[d]) continue;
        int dep[4];
        intra_deps(fp, d, dep);
        if (dep[0] != sb && dep[1] != sb && dep[2] != sb && dep[3] != sb) continue;
        if (__hip_atomic_fetch_add(&cnt[d], -1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == 1) queue_push(q, f << 16 | d);
      }
    }
    __syncthreads();
  }
}

#endif
