/* Loop-restoration parameter search on gfx950 (behaviour of lr_select,
 * src/lr_search.c:235-359): per restoration unit NONE, a separable
 * least-squares Wiener fit refined greedily tap by tap, and the 16
 * self-guided sets with least-squares projection weights; the smallest
 * 16 * SSE + lambda * bits wins.
 *
 * The choice of a unit depends on the previous unit of its plane only
 * through the subexp references of the coded parameters (bit counts), so:
 *   k_lr_fit    three workgroups per unit, all units at once: the SSE of NONE,
 *               the Wiener fit and its greedy refinement under the default
 *               reference; each half of the self-guided sets' weights and SSE;
 *   k_lr_chain  one workgroup per plane makes the choices in order with the
 *               true references. The refinement's SSEs do not depend on the
 *               reference, so a unit's refinement is replayed from its
 *               recorded SSEs, and done again only if a step of the replay
 *               decides otherwise than the record;
 *   k_lr_path   one workgroup per unit: the refinement of the units left
 *               after several such, between two launches of the chain.
 * The Wiener fit is FP64 and its rounded result decides the coded taps: it
 * accumulates in the reference's order (block by block, sample by sample,
 * one lane per accumulator) with the reference's operand order, and this
 * file is compiled without floating-point contraction. Every other sum is
 * an exact integer. */
#include "dev_common.h"
#include "internal.h"

#include <climits>
#pragma clang fp contract(off)

#define LR_PITCH 104   /* unit width (<= 95) + 6 halo columns, rounded up (a multiple of 4) */
#define LR_ROWS 144    /* unit rows (<= 103) + 6 halo rows per stripe segment (<= 4), + the rows a task reads past its last */
#define LR_MAXSEG 4
#define LR_MAXPX (104 * 96)
#define LR_T 256       /* threads per workgroup */
#define LR_CH 16       /* rows of a column task */
#define LR_NM (LR_CH + 6)
#define LR_CK 64       /* columns of a fit chunk: one block row's columns, one per lane */
#define LR_PS 258      /* products per accumulator and chunk (4 x 64), padded off a multiple of the LDS banks */

struct LrGeo {
  int p, sub, x0, x1, y0, y1, endX, endY;
  int nseg;
  int segY0[LR_MAXSEG], segY1[LR_MAXSEG], segS0[LR_MAXSEG], segS1[LR_MAXSEG], segBase[LR_MAXSEG];
  int bw, bh, nbr, nbc;
};

/* A unit's samples, and the refinement's working set. */
struct LrUnitLds {
  alignas(16) uint8_t img[LR_ROWS * LR_PITCH]; /* stripe-resolved source samples (get_source_sample) per segment */
  uint8_t srcu[LR_MAXPX];                      /* the unit's samples of the source frame, row stride = unit width */
  int redi[2][LR_T / 64][3];
  int wb[18]; /* bits of the fitted tap - 1, + 0, + 1 under the incoming reference */
};
/* Working set of the workgroup searching one unit. */
struct LrLds : LrUnitLds {
  union {
    struct {
      alignas(16) int16_t f0[LR_MAXPX], f1[LR_MAXPX]; /* self-guided filter outputs, 16 per 4x4 block */
    } sg;
    struct {
      alignas(16) double pr[2][9][LR_PS]; /* a chunk's products per accumulator, in sample order (two chunks in flight) */
      double v[2][2][LR_CK + 8];          /* per producer wave: vertical 7-tap sums of its rows */
    } wf;
  } u;
  long long red[2][LR_T / 64][5];
  int sse[8][LR_T / 64];
  double acc[12];
  double sol[4];
  int sums[12][LR_T / 64];
  int itmp[2];
  int xtab[256]; /* a of the self-guided filter by z (7.17.3) */
};
__shared__ LrLds gLr;
__shared__ uint8_t gBits[16 + 32 + 64 + 128]; /* subexp bits by recentred value: Wiener taps 0 .. 2, projection weights */

/* What the refinement of a unit evaluated, per tap it tried ([pass * 3 + j]):
 * the SSE of the taps it came with, and of that tap - 1 and + 1. A unit has
 * at most 95 x 103 samples, so an SSE fits 32 bits. */
struct LrTrace {
  uint32_t cur[6], m[6], p[6];
};

/* Where a plane's chain stands between its launches. */
struct LrChain {
  int start; /* next unit (plane index) to decide */
  int done, used, nrerun;
  int ref[6], refX[2]; /* running references */
};

/* Per-unit search state between the kernels. */
struct LrUnitStat {
  uint32_t sseNone;
  uint32_t sseSgr[16];
  int xqd[16][2];
  int w0[6];    /* fitted Wiener taps: [pass * 3 + j] */
  int wStar[6]; /* the taps the refinement arrived at */
  LrTrace tr;
  LrChain chain; /* of the plane, in its first unit */
};

DEVI int lr_stripe_row(int k, int sub) { return (64 * k - 8) >> sub; }

/* Pixel bounds of unit u and its stripe segments (the 4x4 blocks of
 * lr_block_setup, src/kernels/k_lr.h:28-45, whose unit is u). */
DEVI void lr_geo(const Mav1FrameParams &fp, int u, LrGeo &g) {
  const int p = u >= fp.lr_unit_off[2] ? 2 : u >= fp.lr_unit_off[1] ? 1 : 0;
  const int l = u - fp.lr_unit_off[p], ucols = fp.lr_unit_cols[p], urows = fp.lr_unit_rows[p];
  const int ur = l / ucols, uc = l - (l / ucols) * ucols, sub = p > 0;
  g.p = p;
  g.sub = sub;
  g.endX = ((fp.frame_w + sub) >> sub) - 1;
  g.endY = ((fp.frame_h + sub) >> sub) - 1;
  g.x0 = uc * 64;
  g.x1 = uc == ucols - 1 ? g.endX + 1 : d_min((uc + 1) * 64, g.endX + 1);
  const int off = 8 >> sub;
  g.y0 = d_max(0, ur * 64 - off);
  g.y1 = ur == urows - 1 ? g.endY + 1 : d_min((ur + 1) * 64 - off, g.endY + 1);
  g.bw = 4 >> sub;
  g.bh = 4 >> sub;
  g.nbr = (g.y1 - g.y0 + g.bh - 1) / g.bh;
  g.nbc = (g.x1 - g.x0 + g.bw - 1) / g.bw;
  /* unrolled, every index a constant: the arrays stay in registers (the
   * fields of segments past nseg are never read) */
  int k = ((g.y0 << sub) + 8) / 64, base = 0, y = g.y0;
  g.nseg = 0;
#pragma unroll
  for (int i = 0; i < LR_MAXSEG; i++, k++) {
    const int s0 = lr_stripe_row(k, sub), s1 = lr_stripe_row(k + 1, sub) - 1;
    const int a = d_max(y, s0), b = d_min(g.y1, s1 + 1);
    g.segY0[i] = a;
    g.segY1[i] = b;
    g.segS0[i] = s0;
    g.segS1[i] = s1;
    g.segBase[i] = base;
    if (y < g.y1) {
      base += (b - a + 6) * LR_PITCH;
      g.nseg++;
      y = b;
    }
  }
}

/* v[s] by selects over values, so that a run-time segment index does not
 * move the arrays to scratch memory (a select over the array's own
 * elements would be folded back into an indexed load). */
DEVI int lr_pick(int v0, int v1, int v2, int v3, int s) { return s == 0 ? v0 : s == 1 ? v1 : s == 2 ? v2 : v3; }
#define lr_sel(v, s) lr_pick((v)[0], (v)[1], (v)[2], (v)[3], (s))

DEVI int lr_seg_of(const LrGeo &g, int y) { return y < g.segY1[0] ? 0 : y < g.segY1[1] ? 1 : y < g.segY1[2] ? 2 : 3; }

/* get_source_sample (7.17.6) of every sample the unit's filters read, and
 * the unit's source samples: a wave takes every fourth row, a lane a column
 * (and the column 64 further), eight rows' loads in flight. */
DEVI void lr_stage(const Mav1FrameParams &fp, const LrGeo &g, const uint8_t *cdef, const uint8_t *dbk,
                   const uint8_t *src, LrUnitLds &U, int tid) {
  constexpr int NW = LR_T / 64, N = 8;
  const int S = fp.stride[g.p], o = fp.offset[g.p], w = g.x1 - g.x0 + 6, uw = g.x1 - g.x0, uh = g.y1 - g.y0;
  const int wave = d_uni(tid >> 6), lane = tid & 63;
  const int c1 = d_min(lane + 64, uw - 1), c0 = d_min(lane, uw - 1);
  for (int r0 = wave; r0 < uh; r0 += NW * N) {
    int v0[N], v1[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
      const uint8_t *row = src + o + (size_t)(g.y0 + d_min(r0 + NW * k, uh - 1)) * S + g.x0;
      v0[k] = row[c0];
      v1[k] = row[c1];
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int r = r0 + NW * k;
      if (r >= uh) break;
      if (lane < uw) U.srcu[r * uw + lane] = (uint8_t)v0[k];
      if (lane + 64 < uw) U.srcu[r * uw + lane + 64] = (uint8_t)v1[k];
    }
  }
  const int x0 = d_clip(0, g.endX, g.x0 - 3 + lane), x1 = d_clip(0, g.endX, g.x0 - 3 + lane + 64);
  for (int s = 0; s < g.nseg; s++) {
    const int sy0 = lr_sel(g.segY0, s), ss0 = lr_sel(g.segS0, s), ss1 = lr_sel(g.segS1, s);
    const int h = lr_sel(g.segY1, s) - sy0 + 6, sb = lr_sel(g.segBase, s);
    for (int r0 = wave; r0 < h; r0 += NW * N) {
      int v0[N], v1[N];
#pragma unroll
      for (int k = 0; k < N; k++) {
        int y = d_clip(0, g.endY, sy0 - 3 + d_min(r0 + NW * k, h - 1));
        const uint8_t *pl = cdef;
        if (y < ss0) {
          y = d_max(ss0 - 2, y);
          pl = dbk;
        } else if (y > ss1) {
          y = d_min(ss1 + 2, y);
          pl = dbk;
        }
        const uint8_t *row = pl + o + (size_t)y * S;
        v0[k] = row[x0];
        v1[k] = row[x1];
      }
#pragma unroll
      for (int k = 0; k < N; k++) {
        const int r = r0 + NW * k;
        if (r >= h) break;
        if (lane < w) U.img[sb + r * LR_PITCH + lane] = (uint8_t)v0[k];
        if (lane + 64 < w) U.img[sb + r * LR_PITCH + lane + 64] = (uint8_t)v1[k];
      }
    }
  }
  __syncthreads();
}

typedef __attribute__((address_space(3))) const uint32_t lds_u32;
typedef short s16x2 __attribute__((ext_vector_type(2)));
DEVI s16x2 lr_s2(int lo, int hi) {
  union {
    uint32_t u;
    s16x2 v;
  } c;
  c.u = ((uint32_t)lo & 0xFFFF) | (uint32_t)hi << 16;
  return c.v;
}

/* One column of LR_CH rows (fewer at the end of a segment): the unit of work
 * of the passes that filter the whole unit. img: the staged sample under the
 * first row's first vertical tap and the first horizontal tap; q: the first
 * row's index in srcu. Rows past n are staged garbage, never used. */
struct LrTask {
  int img, q, n;
};
DEVI int lr_tasks(const LrGeo &g) {
  int k = 0;
#pragma unroll
  for (int s = 0; s < LR_MAXSEG; s++)
    if (s < g.nseg) k += (g.segY1[s] - g.segY0[s] + LR_CH - 1) / LR_CH;
  return k * (g.x1 - g.x0);
}
DEVI LrTask lr_task(const LrGeo &g, int t) {
  const int uw = g.x1 - g.x0;
  int k = t / uw;
  const int c = t - k * uw;
  LrTask T = {0, 0, 0};
#pragma unroll
  for (int s = 0; s < LR_MAXSEG; s++)
    if (s < g.nseg) {
      const int h = g.segY1[s] - g.segY0[s], n = (h + LR_CH - 1) / LR_CH;
      if (k >= 0 && k < n) {
        T.img = g.segBase[s] + k * LR_CH * LR_PITCH + c;
        T.q = (g.segY0[s] - g.y0 + k * LR_CH) * uw + c;
        T.n = d_min(LR_CH, h - k * LR_CH);
      }
      k -= n;
    }
  return T;
}
/* The task's source samples, four rows per word (0 past n). */
DEVI void lr_task_src(const LrUnitLds &U, const LrTask &T, int uw, uint32_t sv[LR_CH / 4]) {
#pragma unroll
  for (int i = 0; i < LR_CH / 4; i++) sv[i] = 0;
#pragma unroll
  for (int r = 0; r < LR_CH; r++) {
    const uint32_t v = U.srcu[T.q + d_min(r, T.n - 1) * uw];
    sv[r >> 2] |= v << (8 * (r & 3));
  }
}
/* The seven samples of a staged row from byte `at` on: lo = samples 0 .. 3,
 * hi = samples 4 .. 6 and one more. */
DEVI void lr_row7(const LrUnitLds &U, int at, uint32_t &lo, uint32_t &hi) {
  const lds_u32 *w = (const lds_u32 *)(U.img + (at & ~3));
  const uint32_t w0 = w[0], w1 = w[1], w2 = w[2];
  lo = __builtin_amdgcn_alignbyte(w1, w0, at & 3);
  hi = __builtin_amdgcn_alignbyte(w2, w1, at & 3);
}

/* ---- subexp bit counts (lr_search.c:18-79) ---- */
/* The recentred value of v under reference r, both in 0 .. mx - 1 (by selects
 * and arithmetic: every lane takes its own case). */
DEVI int lr_recentred(int mx, int r, int v) {
  const bool flip = 2 * r > mx;
  const int a = flip ? mx - 1 - r : r, b = flip ? mx - 1 - v : v, d = b - a;
  return b > 2 * a ? b : (d * 2) ^ (d >> 31); /* 2 d, or - 2 d - 1 below 0 */
}
DEVI int lr_subexp_bits(int mx, int k, int x) {
  int bits = 0, mk = 0;
  for (int i = 0;; i++) {
    const int b2 = i ? k + i - 1 : k, a = 1 << b2;
    if (mx <= mk + 3 * a) {
      const int n = mx - mk, w = d_floorlog2((unsigned)n) + 1, m = (1 << w) - n;
      return bits + (x - mk < m ? w - 1 : w);
    }
    bits++;
    if (x < mk + a) return bits + b2;
    mk += a;
  }
}
/* The bits of every recentred value: ranges of the three Wiener taps and of
 * the projection weights. */
DEVI void lr_bits_init(int tid) {
  for (int q = tid; q < 16 + 32 + 64 + 128; q += LR_T) {
    const int j = q < 16 ? 0 : q < 48 ? 1 : q < 112 ? 2 : 3, x = q - (j == 0 ? 0 : j == 1 ? 16 : j == 2 ? 48 : 112);
    const int mx = 16 << j, k = j < 3 ? Wiener_Taps_K[j] : SGRPROJ_PRJ_SUBEXP_K;
    gBits[q] = (uint8_t)lr_subexp_bits(mx, k, x);
  }
}
static_assert(LR_T >= 240, "lr_bits_init");
DEVI int lr_tap_bits(int j, int ref, int v) {
  const int lo = Wiener_Taps_Min[j], mx = 16 << j;
  return gBits[(j == 0 ? 0 : j == 1 ? 16 : 48) + lr_recentred(mx, ref - lo, v - lo)];
}
DEVI int lr_xqd_bits(int i, int ref, int v) {
  const int lo = Sgrproj_Xqd_Min[i];
  return gBits[112 + lr_recentred(128, ref - lo, v - lo)];
}
DEVI long long lr_rd(int lambda, long long sse, int bits) { return sse * 16 + (long long)lambda * bits; }

/* ---- the refinement of the Wiener taps ---- */
/* Horizontal pass of taps hw over the task's rows. acc[t] receives the
 * 7-tap sum of row t plus the rounding term: the outer taps as signed bytes
 * times (sample - 128) on the dot products, the centre tap by itself. With
 * DELTA, d[t] receives what one more of tap j (and two less of the centre)
 * adds to it. */
template <bool DELTA>
DEVI void lr_hsum(const LrUnitLds &U, const LrTask &T, const int *hw, int j, int acc[LR_NM], int d[LR_NM]) {
  const int h0 = hw[0], h1 = hw[1], h2 = hw[2], hc = 128 - 2 * (h0 + h1 + h2);
  const int t0 = (h0 & 255) | (h1 & 255) << 8 | (h2 & 255) << 16, t1 = (h2 & 255) | (h1 & 255) << 8 | (h0 & 255) << 16;
  const int init = 256 * (h0 + h1 + h2) + 4;
  const int u0 = 1 << (8 * j), u1 = 1 << (8 * (2 - j));
#pragma unroll
  for (int t = 0; t < LR_NM; t++) {
    uint32_t lo, hi;
    lr_row7(U, T.img + t * LR_PITCH, lo, hi);
    const int l = (int)(lo ^ 0x80808080u), h = (int)(hi ^ 0x80808080u), c = (int)(lo >> 24);
    acc[t] = __builtin_amdgcn_sdot4(h, t1, __builtin_amdgcn_sdot4(l, t0, init, false), false) + __mul24(c, hc);
    if constexpr (DELTA) d[t] = __builtin_amdgcn_sdot4(h, u1, __builtin_amdgcn_sdot4(l, u0, 256, false), false) - 2 * c;
  }
}
/* Rows t and t + 1 of the rounded horizontal pass as a pair of 16-bit values. */
DEVI int lr_mid1(int acc) { return d_clip(-2048, 8191 - 2048, acc >> 3); }
DEVI void lr_pairs(const int m[LR_NM], s16x2 p[LR_NM - 1]) {
#pragma unroll
  for (int t = 0; t < LR_NM - 1; t++) p[t] = lr_s2(m[t], m[t + 1]);
}
/* Sum of seven vertical taps (a b c e c b a) from row r of the pairs on. */
struct LrV {
  s16x2 ab, ce, cb, a;
};
DEVI LrV lr_vtaps(int a, int b, int c, int e) { return {lr_s2(a, b), lr_s2(c, e), lr_s2(c, b), lr_s2(0, a)}; }
DEVI int lr_vsum(const s16x2 *p, int r, const LrV &v, int init) {
  int s = __builtin_amdgcn_sdot2(p[r], v.ab, init, false);
  s = __builtin_amdgcn_sdot2(p[r + 2], v.ce, s, false);
  s = __builtin_amdgcn_sdot2(p[r + 4], v.cb, s, false);
  return __builtin_amdgcn_sdot2(p[r + 5], v.a, s, false);
}
/* Squared error of the task's row r (0 past its last). */
DEVI int lr_sq(const LrTask &T, int r, int acc, const uint32_t *sv) {
  int d = d_clip1(acc >> 11) - (int)((sv[r >> 2] >> (8 * (r & 3))) & 255);
  d = r < T.n ? d : 0;
  return __mul24(d, d);
}

/* A tap's step: - 1 if that is cheaper than the taps it came with (SSE cur),
 * else + 1 if that is, else 0. sm, sp: SSE of the neighbours; b0 .. b2: bits
 * of the tap - 1, + 0, + 1 (the other taps' bits are on both sides). */
DEVI int lr_step(int lambda, int j, int w, uint32_t cur, uint32_t sm, uint32_t sp, int b0, int b1, int b2) {
  const long long c = lr_rd(lambda, cur, b1);
  const bool dn = (w > Wiener_Taps_Min[j]) & (lr_rd(lambda, sm, b0) < c);
  const bool up = (w < Wiener_Taps_Max[j]) & (lr_rd(lambda, sp, b2) < c);
  return dn ? -1 : up ? 1 : 0;
}

/* Greedy +-1 refinement of each coded tap (lr_search.c:283-301) from the
 * taps in w (updated in place) with incoming reference ref; *tr receives the
 * SSEs. Needs the staged samples and the bits table. Every thread gets the
 * same.
 * The reference tries tap - 1, then tap + 1 of what that left. After an
 * accepted - 1, + 1 gives back the taps before at their larger cost, so both
 * neighbours are always taken from the same taps and are evaluated together:
 * one tap more adds (left + right - 2 centre) samples to a 7-tap sum, so the
 * two candidates share the sum of the current taps. A thread holds a column
 * of rows in registers: the vertical taps' rounds read nothing but the
 * source samples.
 * Bound by VALU issue; one barrier per tap, about 40k cycles for a 64x64
 * unit. Candidate by candidate over a horizontal pass in LDS it took more
 * than twice that. */
DEVI void lr_refine(int lambda, const LrGeo &g, LrUnitLds &U, int *w, const int *ref, LrTrace *tr, int tid) {
  const int uw = g.x1 - g.x0, nt = lr_tasks(g), first = g.p ? 1 : 0, wave = tid >> 6;
  if (tid < 18) {
    const int k = tid / 3, j = k % 3;
    int wk = 0, rk = 0; /* by selects, as below: the taps stay in registers */
#pragma unroll
    for (int i = 0; i < 6; i++)
      if (i == k) {
        wk = w[i];
        rk = ref[i];
      }
    U.wb[tid] = j < first ? 0
                            : lr_tap_bits(j, rk, d_clip(Wiener_Taps_Min[j], Wiener_Taps_Max[j], wk + tid % 3 - 1));
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 6; k++) tr->cur[k] = tr->m[k] = tr->p[k] = 0;
  int sse = 0;
  int par = 0;
  bool start = true;
  LrTask T = lr_task(g, tid);
  int m[LR_NM];
  s16x2 p[LR_NM - 1];
  uint32_t sv[LR_CH / 4] = {};
#pragma unroll 1
  for (int pass = 0; pass < 2; pass++)
#pragma unroll 1
    for (int j = first; j < 3; j++) {
      int e0 = 0, em = 0, ep = 0;
      const int vc = 128 - 2 * (w[0] + w[1] + w[2]);
      const LrV V = lr_vtaps(w[0], w[1], w[2], vc);
      if (pass == 0) {
        /* D: + 1 at taps j and 6 - j, - 2 at the centre */
        const LrV D = lr_vtaps(j == 0, j == 1, j == 2, -2);
        for (int t = tid; t < nt; t += LR_T) {
          if (start || nt > LR_T) {
            T = lr_task(g, t);
            lr_task_src(U, T, uw, sv);
            lr_hsum<false>(U, T, w + 3, 0, m, m);
#pragma unroll
            for (int i = 0; i < LR_NM; i++) m[i] = lr_mid1(m[i]);
            lr_pairs(m, p);
          }
#pragma unroll
          for (int r = 0; r < LR_CH; r++) {
            const int a = lr_vsum(p, r, V, 1 << 10), d = lr_vsum(p, r, D, 0);
            if (start) e0 += lr_sq(T, r, a, sv);
            em += lr_sq(T, r, a - d, sv);
            ep += lr_sq(T, r, a + d, sv);
          }
        }
      } else {
        for (int t = tid; t < nt; t += LR_T) {
          if (nt > LR_T) {
            T = lr_task(g, t);
            lr_task_src(U, T, uw, sv);
          }
          int d[LR_NM], x[LR_NM];
          lr_hsum<true>(U, T, w + 3, j, m, d);
#pragma unroll
          for (int i = 0; i < LR_NM; i++) x[i] = lr_mid1(m[i] - d[i]);
          lr_pairs(x, p);
#pragma unroll
          for (int r = 0; r < LR_CH; r++) em += lr_sq(T, r, lr_vsum(p, r, V, 1 << 10), sv);
#pragma unroll
          for (int i = 0; i < LR_NM; i++) x[i] = lr_mid1(m[i] + d[i]);
          lr_pairs(x, p);
#pragma unroll
          for (int r = 0; r < LR_CH; r++) ep += lr_sq(T, r, lr_vsum(p, r, V, 1 << 10), sv);
        }
      }
      e0 = wave_sum_dpp(e0);
      em = wave_sum_dpp(em);
      ep = wave_sum_dpp(ep);
      if ((tid & 63) == 0) {
        U.redi[par][wave][0] = e0;
        U.redi[par][wave][1] = em;
        U.redi[par][wave][2] = ep;
      }
      __syncthreads();
      int s0 = 0, sm = 0, sp = 0;
#pragma unroll
      for (int k = 0; k < LR_T / 64; k++) {
        s0 += U.redi[par][k][0];
        sm += U.redi[par][k][1];
        sp += U.redi[par][k][2];
      }
      par ^= 1;
      const int k = pass * 3 + j;
      if (start) sse = s0;
      start = false;
      int wk = 0;
#pragma unroll
      for (int i = 0; i < 6; i++) {
        wk = i == k ? w[i] : wk;
        tr->cur[i] = i == k ? (uint32_t)sse : tr->cur[i];
        tr->m[i] = i == k ? (uint32_t)sm : tr->m[i];
        tr->p[i] = i == k ? (uint32_t)sp : tr->p[i];
      }
      const int d = lr_step(lambda, j, wk, sse, sm, sp, U.wb[3 * k], U.wb[3 * k + 1], U.wb[3 * k + 2]);
      wk += d;
      sse = d < 0 ? sm : d > 0 ? sp : sse;
#pragma unroll
      for (int i = 0; i < 6; i++) w[i] = i == k ? wk : w[i];
    }
}

DEVI void lr_record(LrUnitStat &st, const int *w, const LrTrace &tr) {
#pragma unroll
  for (int k = 0; k < 6; k++) st.wStar[k] = w[k];
  st.tr = tr;
}
/* ---- the Wiener fit ---- */
/* Gaussian elimination with partial pivoting (lr_search.c:98-129); rows
 * change place by selects, so that the matrix stays in registers. */
template <int N>
DEVI int lr_solve(double (&M)[N][N], double (&v)[N], double (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; i++) {
    int piv = i;
    double pa = fabs(M[i][i]);
#pragma unroll
    for (int r = i + 1; r < N; r++)
      if (fabs(M[r][i]) > pa) {
        piv = r;
        pa = fabs(M[r][i]);
      }
    if (pa < 1e-9) return 0;
#pragma unroll
    for (int r = i + 1; r < N; r++) {
      const bool sw = piv == r;
#pragma unroll
      for (int k = 0; k < N; k++) {
        const double t = M[i][k];
        M[i][k] = sw ? M[r][k] : t;
        M[r][k] = sw ? t : M[r][k];
      }
      const double t = v[i];
      v[i] = sw ? v[r] : t;
      v[r] = sw ? t : v[r];
    }
#pragma unroll
    for (int r = i + 1; r < N; r++) {
      const double f = M[r][i] / M[i][i];
#pragma unroll
      for (int k = i; k < N; k++) M[r][k] -= f * M[i][k];
      v[r] -= f * v[i];
    }
  }
#pragma unroll
  for (int i = N - 1; i >= 0; i--) {
    double s = v[i];
#pragma unroll
    for (int k = i + 1; k < N; k++) s -= M[i][k] * x[k];
    x[i] = s / M[i][i];
  }
  return 1;
}

/* The accumulators of a fit with NC taps: the upper triangle of the matrix
 * row by row (its products commute, so the lower one is the same), then the
 * right-hand side. */
template <int NC>
constexpr int lr_macc(int a, int b) {
  return a <= b ? a * NC - a * (a - 1) / 2 + b - a : lr_macc<NC>(b, a);
}

/* SSE of NONE and the first solve's sums (a vertical fit under the identity
 * horizontal filter): every fit term is then an integer (|phi| <= 510,
 * |target| <= 255), so every product and partial sum of the reference's FP64
 * accumulation is an integer below 2^53 and exact, whatever the order.
 * All lanes sum their samples in int32 (<= 48 samples x 510^2 each, so a
 * wave's sum fits too); the sums land in gLr.acc as doubles. */
template <int NC>
DEVI uint32_t lr_wf_exact(const LrGeo &g, int tid) {
  constexpr int FIRST = 3 - NC, NP = NC * (NC + 1) / 2 + NC;
  const int uw = g.x1 - g.x0, nt = lr_tasks(g), wave = tid >> 6;
  int sum[NP + 1];
#pragma unroll
  for (int i = 0; i <= NP; i++) sum[i] = 0;
  for (int t = tid; t < nt; t += LR_T) {
    const LrTask T = lr_task(g, t);
    int Z[LR_NM];
#pragma unroll
    for (int i = 0; i < LR_NM; i++) Z[i] = gLr.img[T.img + 3 + i * LR_PITCH];
    uint32_t sv[LR_CH / 4];
    lr_task_src(gLr, T, uw, sv);
#pragma unroll
    for (int r = 0; r < LR_CH; r++) {
      int ph[NC + 1];
#pragma unroll
      for (int a = 0; a < NC; a++) {
        ph[a] = Z[r + FIRST + a] + Z[r + 6 - FIRST - a] - 2 * Z[r + 3];
        ph[a] = r < T.n ? ph[a] : 0;
      }
      ph[NC] = (int)((sv[r >> 2] >> (8 * (r & 3))) & 255) - Z[r + 3];
      ph[NC] = r < T.n ? ph[NC] : 0;
#pragma unroll
      for (int a = 0; a < NC; a++) {
#pragma unroll
        for (int b = a; b < NC; b++) sum[lr_macc<NC>(a, b)] += __mul24(ph[a], ph[b]);
        sum[NP - NC + a] += __mul24(ph[a], ph[NC]);
      }
      sum[NP] += __mul24(ph[NC], ph[NC]);
    }
  }
#pragma unroll
  for (int i = 0; i <= NP; i++) {
    const int v = wave_sum_dpp(sum[i]);
    if ((tid & 63) == 0) gLr.sums[i][wave] = v;
  }
  __syncthreads();
  if (tid < NP) {
    long long t = 0;
#pragma unroll
    for (int w = 0; w < LR_T / 64; w++) t += gLr.sums[tid][w];
    gLr.acc[tid] = (double)t;
  }
  uint32_t sse = 0;
#pragma unroll
  for (int w = 0; w < LR_T / 64; w++) sse += (uint32_t)gLr.sums[NP][w];
  return sse;
}

/* The 7-tap sum of samples lo / hi under filter f in the reference's order. */
DEVI double lr_sum7(const double *f, uint32_t lo, uint32_t hi) {
  double s = 0;
#pragma unroll
  for (int t = 0; t < 7; t++) s += f[t] * (double)(t < 4 ? (lo >> (8 * t)) & 255 : (hi >> (8 * (t - 4))) & 255);
  return s;
}
/* Position of sample (r, x) of block j of a chunk: a block's samples are
 * apart by constants, and a row of samples spreads over the LDS banks (in
 * the order of the samples the stores met in an eighth of them). */
template <int BS>
constexpr DEVI int lr_wf_pos(int j, int r, int x) {
  return ((r * (BS / 2) + (x >> 1)) * (LR_CK / BS) + j) * 2 + (x & 1);
}
/* The products of one sample's fit terms (lr_search.c:150-160): phi[a] =
 * Z[a] + Z[6 - a] - 2 Z[3], target src - Z[3]; zeros where the block has no
 * sample, which leave the sums unchanged (they start at + 0). */
template <int NC>
DEVI void lr_wf_products(const double *Z, double src, bool in, int buf, int at) {
  constexpr int FIRST = 3 - NC, NP = NC * (NC + 1) / 2 + NC;
  double ph[NC];
#pragma unroll
  for (int a = 0; a < NC; a++) ph[a] = Z[FIRST + a] + Z[6 - FIRST - a] - 2 * Z[3];
  const double tg = src - Z[3];
#pragma unroll
  for (int a = 0; a < NC; a++) {
#pragma unroll
    for (int b = a; b < NC; b++) gLr.u.wf.pr[buf][lr_macc<NC>(a, b)][at] = in ? ph[a] * ph[b] : 0.0;
    gLr.u.wf.pr[buf][NP - NC + a][at] = in ? ph[a] * tg : 0.0;
  }
}
/* A value from one row of 16 lanes to the next in the order 0, 1, 3, 2
 * (step 0 .. 3: into row 1, 3, 2, 0); the other rows get anything. */
template <int STEP>
DEVI double lr_row_next(double v) {
  union {
    double d;
    unsigned u[2];
  } c;
  c.d = v;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    if constexpr (STEP & 1) c.u[i] = __builtin_amdgcn_permlane32_swap(c.u[i], c.u[i], false, false)[STEP >> 1];
    else c.u[i] = __builtin_amdgcn_permlane16_swap(c.u[i], c.u[i], false, false)[STEP >> 1];
  }
  return c.d;
}
/* acc plus the products of ns groups of 64 samples in order; acc of
 * accumulator a is held by lane a. Each row of 16 lanes loads 16 consecutive
 * samples (one 4x4 block or four 2x2 blocks) of the group's 64 in eight
 * loads, and the running sums pass from row to row, in which the row's
 * samples are added: with every sample loaded by row 0 the adding wave
 * issued four times the loads, and a sample took 14 cycles (an addition
 * waits 8 for the one before). */
template <int BS>
DEVI double lr_wf_chain(const double *row, int ns, double acc, int lane) {
  typedef double d2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) const d2 lds_d2;
  constexpr int G = 16 / (BS * BS); /* blocks of 16 samples */
  const int r = lane >> 4;
  const lds_d2 *p = (const lds_d2 *)row + (r ^ (r >> 1)) * G;
  d2 x[8], y[8];
  auto load = [&](d2 (&v)[8], int b) {
    const lds_d2 *q = p + b * (4 * G);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int e = 2 * k;
      v[k] = q[lr_wf_pos<BS>(e / (BS * BS), e / BS % BS, e % BS) / 2];
    }
  };
  auto add = [&](const d2 (&v)[8]) {
    auto row16 = [&]() {
#pragma unroll
      for (int k = 0; k < 8; k++) {
        acc += v[k].x;
        acc += v[k].y;
      }
    };
    row16();
    acc = lr_row_next<0>(acc);
    row16();
    acc = lr_row_next<1>(acc);
    row16();
    acc = lr_row_next<2>(acc);
    row16();
    acc = lr_row_next<3>(acc);
  };
  load(x, 0);
  for (int b = 0; b < ns; b += 2) {
    load(y, d_min(b + 1, ns - 1));
    __builtin_amdgcn_sched_barrier(0);
    add(x);
    __builtin_amdgcn_sched_barrier(0);
    load(x, d_min(b + 2, ns - 1));
    __builtin_amdgcn_sched_barrier(0);
    if (b + 1 < ns) add(y);
    __builtin_amdgcn_sched_barrier(0);
  }
  return acc;
}

/* The sums of a later solve: the products run over the unit's samples in the
 * reference's order (blocks of BS x BS of a block row, samples of a block),
 * in chunks of up to LR_CK columns of a block row. Waves 1 and 2 each make
 * the products of half of a chunk's rows, one column per lane; wave 0 adds
 * the chunk before, one lane per accumulator. Vertical fit (VERT): f is the
 * horizontal filter, and a lane keeps the filtered rows of its column from
 * block row to block row; else f is the vertical filter. */
template <int NC, int BS, bool VERT>
DEVI void lr_wf_sums(const LrGeo &g, const double *f, int tid) {
  constexpr int NP = NC * (NC + 1) / 2 + NC, RP = BS / 2, W = RP + 6;
  const int uw = g.x1 - g.x0, ncg = (uw + LR_CK - 1) / LR_CK, nch = g.nbr * ncg;
  const int wave = d_uni(tid >> 6), lane = tid & 63, r0 = RP * (wave - 1);
  double acc = 0, H[2][W];
#pragma unroll
  for (int i = 0; i < W; i++) H[0][i] = H[1][i] = 0;
  int br = 0, cg = 0, pn = 0; /* the chunk to make; groups of 64 samples of the one before */
  for (int i = 0; i <= nch; i++) {
    const int y0 = g.y0 + br * BS, s = lr_seg_of(g, y0), h = d_min(BS, g.endY - y0 + 1), cw = d_min(LR_CK, uw - cg * LR_CK);
    const int cwb = (cw + 64 / BS - 1) & ~(64 / BS - 1); /* columns in whole groups of 64 samples */
    if (wave == 0) {
      if (i > 0) acc = lr_wf_chain<BS>(gLr.u.wf.pr[(i - 1) & 1][d_min(lane & 15, NP - 1)], pn, acc, lane);
    } else if (wave <= 2 && i < nch) {
      const int c = d_min(lane, cw - 1), cc = cg * LR_CK + c;
      const int row0 = lr_sel(g.segBase, s) + (y0 - lr_sel(g.segY0, s) + r0) * LR_PITCH; /* the first row's first tap */
      const int at = lr_wf_pos<BS>(lane / BS, 0, lane % BS); /* of the column's sample in the block row's first row */
      const uint8_t *sp = gLr.srcu + (y0 - g.y0 + r0) * uw + cc;
      if constexpr (VERT) {
        const bool fresh = br == 0 || y0 == lr_sel(g.segY0, s);
        auto make = [&](double (&Hc)[W]) {
          if (fresh) {
#pragma unroll
            for (int t = 0; t < W - 2 * RP; t++) {
              uint32_t lo, hi;
              lr_row7(gLr, row0 + t * LR_PITCH + cc, lo, hi);
              Hc[t] = lr_sum7(f, lo, hi);
            }
          } else {
#pragma unroll
            for (int t = 0; t < W - 2 * RP; t++) Hc[t] = Hc[t + 2 * RP];
          }
#pragma unroll
          for (int t = W - 2 * RP; t < W; t++) {
            uint32_t lo, hi;
            lr_row7(gLr, row0 + t * LR_PITCH + cc, lo, hi);
            Hc[t] = lr_sum7(f, lo, hi);
          }
#pragma unroll
          for (int r = 0; r < RP; r++)
            if (lane < cwb)
              lr_wf_products<NC>(Hc + r, (double)sp[d_min(r, h - 1 - r0) * uw], r0 + r < h && lane < cw, i & 1,
                                 at + (r0 + r) * LR_CK);
        };
        if (cg == 0) make(H[0]);
        else make(H[1]);
      } else {
        /* vertical sums of the chunk's columns and the three on either side */
        double(*v)[LR_CK + 8] = gLr.u.wf.v[wave - 1];
        const int nv = cw + 6, c0 = cg * LR_CK + d_min(lane, nv - 1);
        int b[RP + 6];
#pragma unroll
        for (int t = 0; t < RP + 6; t++) b[t] = gLr.img[row0 + t * LR_PITCH + c0];
#pragma unroll
        for (int r = 0; r < RP; r++) {
          double sum = 0;
#pragma unroll
          for (int t = 0; t < 7; t++) sum += f[t] * (double)b[r + t];
          v[r][d_min(lane, nv - 1)] = sum;
        }
        if (nv > 64 && lane < 6 * RP) {
          const int r = lane / 6, e = 64 + lane - 6 * r, ce = d_min(e, nv - 1);
          const int at = row0 + r * LR_PITCH + cg * LR_CK + ce;
          double sum = 0;
#pragma unroll
          for (int t = 0; t < 7; t++) sum += f[t] * (double)(int)gLr.img[at + t * LR_PITCH];
          v[r][ce] = sum;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int r = 0; r < RP; r++) {
          double Z[7];
#pragma unroll
          for (int a = 0; a < 7; a++) Z[a] = v[r][c + a];
          if (lane < cwb)
            lr_wf_products<NC>(Z, (double)sp[d_min(r, h - 1 - r0) * uw], r0 + r < h && lane < cw, i & 1,
                               at + (r0 + r) * LR_CK);
        }
      }
    }
    pn = cwb * BS / 64;
    if (++cg == ncg) {
      cg = 0;
      br++;
    }
    __syncthreads();
  }
  if (wave == 0 && lane < NP) gLr.acc[lane] = acc;
}

/* Separable least-squares Wiener fit (lr_search.c:132-180): four
 * alternating solves. The first solve's sums are exact integers
 * (lr_wf_exact), which also gives the SSE of NONE (returned); each later
 * solve's sums are ordered FP64 sums (lr_wf_sums).
 * Bound by the serial chain of FP64 additions, 3 x 4096 for a 64x64 unit at
 * 10 cycles each (lr_wf_chain): the products are made by other waves, because
 * with the multiplication and both operands' loads in the adding lane a
 * sample took 31 cycles. k_lr_fit: 137 us on a 204x116 frame and 400 us on
 * 1920x1080, where it took 309 and 1033 us. */
template <int NC, int BS>
DEVI uint32_t lr_wiener_fit(const LrGeo &g, int *out, int tid) {
  constexpr int FIRST = 3 - NC;
  double fv[7] = {0, 0, 0, 1, 0, 0, 0}, fh[7] = {0, 0, 0, 1, 0, 0, 0};
  uint32_t sseNone = 0;
#pragma unroll 1
  for (int it = 0; it < 4; it++) {
    const bool vert = !(it & 1);
    if (it == 0) sseNone = lr_wf_exact<NC>(g, tid);
    else if (vert) lr_wf_sums<NC, BS, true>(g, fh, tid);
    else lr_wf_sums<NC, BS, false>(g, fv, tid);
    __syncthreads();
    if (tid == 0) {
      double M[NC][NC], V[NC], x[NC];
#pragma unroll
      for (int a = 0; a < NC; a++) {
        V[a] = gLr.acc[NC * (NC + 1) / 2 + a];
        x[a] = 0;
#pragma unroll
        for (int b = 0; b < NC; b++) M[a][b] = gLr.acc[lr_macc<NC>(a, b)];
      }
#pragma unroll
      for (int a = 0; a < NC; a++) M[a][a] += 1e-3;
      gLr.itmp[0] = lr_solve<NC>(M, V, x);
#pragma unroll
      for (int a = 0; a < 3; a++) gLr.sol[a] = a < FIRST ? 0 : x[a < FIRST ? 0 : a - FIRST];
    }
    __syncthreads();
    if (!gLr.itmp[0]) break;
    double sum = 0;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const double v = gLr.sol[a];
      if (vert) fv[a] = fv[6 - a] = v;
      else fh[a] = fh[6 - a] = v;
      sum += v;
    }
    if (vert) fv[3] = 1 - 2 * sum;
    else fh[3] = 1 - 2 * sum;
    __syncthreads();
  }
#pragma unroll
  for (int pass = 0; pass < 2; pass++)
#pragma unroll
    for (int j = 0; j < 3; j++)
      out[pass * 3 + j] =
          j < FIRST ? 0 : d_clip(Wiener_Taps_Min[j], Wiener_Taps_Max[j], (int)lround((pass ? fh[j] : fv[j]) * 128));
  return sseNone;
}

/* ---- the self-guided sets ---- */
/* The filter's a by z: 1 at z = 0, 256 from z = 255, else round(256 z / (z + 1)). */
DEVI void lr_xtab(int tid) {
  for (int z = tid; z < 256; z += LR_T)
    gLr.xtab[z] = z == 0 ? 1 : z == 255 ? 256 : ((z << SGRPROJ_SGR_BITS) + z / 2) / (z + 1);
  __syncthreads();
}
/* Box sums around the 4x4 block whose first staged row and column are at
 * `at` (three above and left of the block): radius 1 at the 6x6 positions
 * (rows -1 .. 4, columns -1 .. 4 of the block), radius 2 at the rows -1, 1
 * and 3. S: the sum, P: n * (sum of squares) - S^2. They do not depend on the
 * set, so a thread keeps them in registers over the sets. */
struct LrBox {
  int S1[36], P1[36], S2[18], P2[18];
};
DEVI void lr_box(int at, LrBox &B) {
  int Q1[36], Q2[18];
#pragma unroll
  for (int i = 0; i < 36; i++) B.S1[i] = Q1[i] = 0;
#pragma unroll
  for (int i = 0; i < 18; i++) B.S2[i] = Q2[i] = 0;
#pragma unroll
  for (int y = 0; y < 9; y++) {
    const lds_u32 *w = (const lds_u32 *)(gLr.img + at + y * LR_PITCH);
    const uint32_t w0 = w[0], w1 = w[1], w2 = w[2];
    int v[10], q[10];
#pragma unroll
    for (int x = 0; x < 10; x++) {
      v[x] = (int)(((x < 4 ? w0 : x < 8 ? w1 : w2) >> (8 * (x & 3))) & 255);
      q[x] = __mul24(v[x], v[x]);
    }
#pragma unroll
    for (int j = 0; j < 6; j++) {
      const int s3 = v[j + 1] + v[j + 2] + v[j + 3], q3 = q[j + 1] + q[j + 2] + q[j + 3];
#pragma unroll
      for (int i = 0; i < 6; i++)
        if (y > i && y < i + 4) {
          B.S1[i * 6 + j] += s3;
          Q1[i * 6 + j] += q3;
        }
      const int s5 = s3 + v[j] + v[j + 4], q5 = q3 + q[j] + q[j + 4];
#pragma unroll
      for (int i = 0; i < 3; i++)
        if (y >= 2 * i && y < 2 * i + 5) {
          B.S2[i * 6 + j] += s5;
          Q2[i * 6 + j] += q5;
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 36; i++) B.P1[i] = Q1[i] * 9 - __mul24(B.S1[i], B.S1[i]);
#pragma unroll
  for (int i = 0; i < 18; i++) B.P2[i] = Q2[i] * 25 - __mul24(B.S2[i], B.S2[i]);
}
/* a and b of a position. P * sc stays below 2^32 - 2^19: P <= 1300500 with
 * sc <= 3236 (radius 1), P <= 10143900 with sc <= 140 (radius 2). */
DEVI void lr_ab(int S, int P, int sc, int one, int &a, int &b) {
  const uint32_t z = (__umul24((uint32_t)P, (uint32_t)sc) + (1u << (SGRPROJ_MTABLE_BITS - 1))) >> SGRPROJ_MTABLE_BITS;
  a = gLr.xtab[z < 255u ? z : 255u];
  b = (__mul24(__mul24((1 << SGRPROJ_SGR_BITS) - a, S), one) + (1 << (SGRPROJ_RECIP_BITS - 1))) >> SGRPROJ_RECIP_BITS;
}
/* The block's filtered samples (7.17.3): radius 2 (weights 6 and 5 on every
 * other row) and radius 1 (weights 4 and 3). px: the block's samples, a row
 * per word. */
DEVI void lr_f2(const LrBox &B, const uint32_t px[4], int sc, int one, int F[16]) {
  int ha[3][4], hb[3][4];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    int a[6], b[6];
#pragma unroll
    for (int j = 0; j < 6; j++) lr_ab(B.S2[i * 6 + j], B.P2[i * 6 + j], sc, one, a[j], b[j]);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      ha[i][j] = 5 * (a[j] + a[j + 1] + a[j + 2]) + a[j + 1];
      hb[i][j] = 5 * (b[j] + b[j + 1] + b[j + 2]) + b[j + 1];
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int u = (int)((px[i] >> (8 * j)) & 255), k = (i + 1) >> 1;
      const int a = (i & 1) ? ha[k][j] : ha[k][j] + ha[k + 1][j], b = (i & 1) ? hb[k][j] : hb[k][j] + hb[k + 1][j];
      const int sh = SGRPROJ_SGR_BITS + ((i & 1) ? 4 : 5) - SGRPROJ_RST_BITS;
      F[i * 4 + j] = (__mul24(a, u) + b + (1 << (sh - 1))) >> sh;
    }
}
DEVI void lr_f1(const LrBox &B, const uint32_t px[4], int sc, int one, int F[16]) {
  int A[6][6], D[6][6];
#pragma unroll
  for (int i = 0; i < 6; i++)
#pragma unroll
    for (int j = 0; j < 6; j++) lr_ab(B.S1[i * 6 + j], B.P1[i * 6 + j], sc, one, A[i][j], D[i][j]);
  constexpr int sh = SGRPROJ_SGR_BITS + 5 - SGRPROJ_RST_BITS;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int va[6], vb[6];
#pragma unroll
    for (int j = 0; j < 6; j++) {
      va[j] = A[i][j] + A[i + 1][j] + A[i + 2][j];
      vb[j] = D[i][j] + D[i + 1][j] + D[i + 2][j];
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      /* 3 everywhere, 1 more on the centre row and column */
      const int a = 3 * (va[j] + va[j + 1] + va[j + 2]) + va[j + 1] + A[i + 1][j] + A[i + 1][j + 2];
      const int b = 3 * (vb[j] + vb[j + 1] + vb[j + 2]) + vb[j + 1] + D[i + 1][j] + D[i + 1][j + 2];
      const int u = (int)((px[i] >> (8 * j)) & 255);
      F[i * 4 + j] = (__mul24(a, u) + b + (1 << (sh - 1))) >> sh;
    }
  }
}
/* Sum over the wave of a value of up to 2^30 in magnitude. */
DEVI long long lr_wave_sum(int v) {
  const int lo = wave_sum_dpp(v & 0xFFFF), hi = wave_sum_dpp(v >> 16);
  return (long long)hi * 65536 + lo;
}

/* The even (half 0) or odd sets of a unit (both halves alike in passes): weights (sgr_fit,
 * lr_search.c:183-231) and SSE. A thread takes a 4x4 block (of luma and
 * chroma alike: stripes and units start at multiples of four rows) with its
 * box sums, samples and source in registers over the sets; units of more
 * than LR_T blocks take them in rounds and build those again per set. The
 * filtered samples wait in LDS for the weights.
 * Bound by VALU issue and the table's LDS reads, about 12k cycles per 64x64
 * unit and set (box sums anew per set and block took about 25k). */
DEVI void lr_sets(const LrGeo &g, int half, LrUnitStat &st, int tid) {
  lr_xtab(tid);
  const int uw = g.x1 - g.x0, uh = g.y1 - g.y0, ncol = (uw + 3) >> 2, nblk = ncol * ((uh + 3) >> 2), wave = tid >> 6;
  LrBox B;
  uint32_t px[4] = {0, 0, 0, 0}, sx[4] = {0, 0, 0, 0};
  int in = 0; /* bit i * 4 + j: the block's sample (i, j) lies in the unit */
  auto pixels = [&](int bi) {
    const int br = bi / ncol, bc = bi - br * ncol, y = g.y0 + br * 4, s = lr_seg_of(g, y);
    const int at = lr_sel(g.segBase, s) + (y - lr_sel(g.segY0, s)) * LR_PITCH + bc * 4;
    const int bw = d_min(4, uw - bc * 4), bh = d_min(4, uh - br * 4);
    in = ((1 << bw) - 1) * 0x1111 & ((1 << (4 * bh)) - 1);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const lds_u32 *w = (const lds_u32 *)(gLr.img + at + (i + 3) * LR_PITCH);
      const uint8_t *sr = gLr.srcu + (br * 4 + d_min(i, bh - 1)) * uw + bc * 4;
      px[i] = __builtin_amdgcn_alignbyte(w[1], w[0], 3);
      sx[i] = sr[0] | (uint32_t)sr[d_min(1, bw - 1)] << 8 | (uint32_t)sr[d_min(2, bw - 1)] << 16 |
              (uint32_t)sr[d_min(3, bw - 1)] << 24;
    }
    return at;
  };
#pragma unroll 1
  for (int k = 0; k < 8; k++) {
    const int set = 2 * k + half;
    /* the radii are 2 (pass 0) and 1 (pass 1), or 0: pass off */
    const int r0 = SGR_PARAM(set, 0), r1 = SGR_PARAM(set, 2);
    int sc[2], one[2];
#pragma unroll
    for (int pass = 0; pass < 2; pass++) {
      const int n = pass ? 9 : 25, n2e = n * n * SGR_PARAM(set, pass * 2 + 1);
      sc[pass] = n2e ? ((1 << SGRPROJ_MTABLE_BITS) + n2e / 2) / n2e : 0;
      one[pass] = ((1 << SGRPROJ_RECIP_BITS) + n / 2) / n;
    }
    int h00 = 0, h01 = 0, h11 = 0, c0 = 0, c1 = 0; /* <= 3 blocks x 16 samples x 4080^2 */
    for (int bi = tid; bi < nblk; bi += LR_T) {
      if (k == 0 || nblk > LR_T) lr_box(pixels(bi), B);
      int F0[16], F1[16];
      if (r0) lr_f2(B, px, sc[0], one[0], F0);
      if (r1) lr_f1(B, px, sc[1], one[1], F1);
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int uu = (int)((px[i] >> (8 * j)) & 255) << SGRPROJ_RST_BITS;
          const int sv = ((int)((sx[i] >> (8 * j)) & 255) << SGRPROJ_RST_BITS) - uu;
          if (!r0) F0[i * 4 + j] = uu;
          if (!r1) F1[i * 4 + j] = uu;
          const int mask = __builtin_amdgcn_sbfe(in, i * 4 + j, 1); /* all ones inside the unit */
          const int e0 = (F0[i * 4 + j] - uu) & mask, e1 = (F1[i * 4 + j] - uu) & mask;
          h00 += __mul24(e0, e0);
          h01 += __mul24(e0, e1);
          h11 += __mul24(e1, e1);
          c0 += __mul24(e0, sv);
          c1 += __mul24(e1, sv);
        }
      int4 *o0 = (int4 *)(gLr.u.sg.f0 + bi * 16), *o1 = (int4 *)(gLr.u.sg.f1 + bi * 16);
      int q0[8], q1[8];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        q0[i] = (F0[2 * i] & 0xFFFF) | F0[2 * i + 1] << 16;
        q1[i] = (F1[2 * i] & 0xFFFF) | F1[2 * i + 1] << 16;
      }
      o0[0] = make_int4(q0[0], q0[1], q0[2], q0[3]);
      o0[1] = make_int4(q0[4], q0[5], q0[6], q0[7]);
      o1[0] = make_int4(q1[0], q1[1], q1[2], q1[3]);
      o1[1] = make_int4(q1[4], q1[5], q1[6], q1[7]);
    }
    /* the five sums in one exchange (two buffers, so one barrier per set);
     * every thread then computes the weights */
    const long long part[5] = {lr_wave_sum(h00), lr_wave_sum(h01), lr_wave_sum(h11), lr_wave_sum(c0), lr_wave_sum(c1)};
    if ((tid & 63) == 0) {
#pragma unroll
      for (int i = 0; i < 5; i++) gLr.red[k & 1][wave][i] = part[i];
    }
    __syncthreads();
    long long tot[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < LR_T / 64; w++)
#pragma unroll
      for (int i = 0; i < 5; i++) tot[i] += gLr.red[k & 1][w][i];
    /* the reference's double sums of integer terms are exact: the same
     * values as these integer sums */
    const double H00 = (double)tot[0], H01 = (double)tot[1], H11 = (double)tot[2], C0 = (double)tot[3], C1 = (double)tot[4];
    double a = 0, bb = 0;
    if (r0 && r1) {
      const double det = H00 * H11 - H01 * H01;
      if (fabs(det) > 1e-9) {
        a = (C0 * H11 - C1 * H01) / det;
        bb = (C1 * H00 - C0 * H01) / det;
      }
    } else if (r0) {
      if (H00 > 0) a = C0 / H00;
    } else if (r1) {
      if (H11 > 0) bb = C1 / H11;
    }
    const int w0q = r0 ? (int)lround(a * (1 << SGRPROJ_PRJ_BITS)) : 0, w2q = (int)lround(bb * (1 << SGRPROJ_PRJ_BITS));
    const int xw0 = d_uni(d_clip(Sgrproj_Xqd_Min[0], Sgrproj_Xqd_Max[0], w0q));
    const int xw1 = d_uni(d_clip(Sgrproj_Xqd_Min[1], Sgrproj_Xqd_Max[1], (1 << SGRPROJ_PRJ_BITS) - xw0 - (r1 ? w2q : 0)));
    const int xw2 = (1 << SGRPROJ_PRJ_BITS) - xw0 - xw1;
    if (tid == 0) {
      st.xqd[set][0] = xw0;
      st.xqd[set][1] = xw1;
    }
    int es = 0; /* <= 48 squared differences of 8-bit samples */
    for (int bi = tid; bi < nblk; bi += LR_T) {
      if (nblk > LR_T) pixels(bi);
      const int4 *o0 = (const int4 *)(gLr.u.sg.f0 + bi * 16), *o1 = (const int4 *)(gLr.u.sg.f1 + bi * 16);
      const int4 v0 = o0[0], v1 = o0[1], u0 = o1[0], u1 = o1[1];
      const int q0[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
      const int q1[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int e = i * 4 + j, uu = (int)((px[i] >> (8 * j)) & 255) << SGRPROJ_RST_BITS;
            const int f0 = (e & 1) ? q0[e >> 1] >> 16 : (int)(int16_t)q0[e >> 1];
            const int f1 = (e & 1) ? q1[e >> 1] >> 16 : (int)(int16_t)q1[e >> 1];
            const int v = __mul24(xw1, uu) + __mul24(xw0, f0) + __mul24(xw2, f1);
            int d = d_clip1(d_round2(v, SGRPROJ_RST_BITS + SGRPROJ_PRJ_BITS)) - (int)((sx[i] >> (8 * j)) & 255);
            d &= __builtin_amdgcn_sbfe(in, e, 1);
            es += __mul24(d, d);
          }
    }
    es = wave_sum_dpp(es);
    if ((tid & 63) == 0) gLr.sse[k][wave] = es;
  }
  __syncthreads();
  if (tid < 8) {
    uint32_t s = 0;
#pragma unroll
    for (int w = 0; w < LR_T / 64; w++) s += (uint32_t)gLr.sse[tid][w];
    st.sseSgr[2 * tid + half] = s;
  }
}

/* Per unit: SSE of NONE, the Wiener fit and its refinement under the default
 * reference, and each self-guided set's weights and SSE. Three workgroups
 * per unit (blockIdx.y), the long serial fits first: NONE and Wiener, the
 * even sets, the odd sets. */
DEVI void lr_fit_body(const Mav1FrameParams &fp, const uint8_t *__restrict__ src, const uint8_t *__restrict__ cdef, const uint8_t *__restrict__ dbk, LrUnitStat *__restrict__ stats, const int u, const int part) {
  const int tid = threadIdx.x;
  LrGeo g;
  lr_geo(fp, u, g);
  lr_stage(fp, g, cdef, dbk, src, gLr, tid);
  LrUnitStat &st = stats[u];
  if (part > 0) {
    lr_sets(g, part - 1, st, tid);
    return;
  }
  lr_bits_init(tid);
  if (tid == 0 && u == fp.lr_unit_off[g.p]) {
    LrChain c = {};
    for (int k = 0; k < 6; k++) c.ref[k] = Wiener_Taps_Mid[k % 3];
    for (int k = 0; k < 2; k++) c.refX[k] = Sgrproj_Xqd_Mid[k];
    st.chain = c;
  }
  int w[6];
  const uint32_t sseNone = g.p ? lr_wiener_fit<2, 2>(g, w, tid) : lr_wiener_fit<3, 4>(g, w, tid);
  int ref[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    ref[k] = Wiener_Taps_Mid[k % 3];
    if (tid == 0) st.w0[k] = w[k];
  }
  if (tid == 0) st.sseNone = sseNone;
  LrTrace tr;
  lr_refine(fp.lambda, g, gLr, w, ref, &tr, tid);
  if (tid == 0) lr_record(st, w, tr);
}
__global__ __launch_bounds__(LR_T) void k_lr_fit(const Mav1FrameParams fp, const uint8_t *__restrict__ src,
                                                 const uint8_t *__restrict__ cdef, const uint8_t *__restrict__ dbk,
                                                 LrUnitStat *__restrict__ stats) {
  lr_fit_body(fp, src, cdef, dbk, stats, blockIdx.x, blockIdx.y);
}

/* Per unit: the refinement under the plane's running reference, for the
 * units from the chain's restart point on (none if it is done). */
DEVI void lr_path_body(const Mav1FrameParams &fp, const uint8_t *__restrict__ src, const uint8_t *__restrict__ cdef, const uint8_t *__restrict__ dbk, LrUnitStat *__restrict__ stats, const int u) {
  __shared__ LrUnitLds U;
  const int tid = threadIdx.x, p = u < fp.lr_unit_off[1] ? 0 : u < fp.lr_unit_off[2] ? 1 : 2;
  const LrChain &cs = stats[fp.lr_unit_off[p]].chain;
  if (cs.done || u - fp.lr_unit_off[p] < cs.start) return;
  LrGeo g;
  lr_geo(fp, u, g);
  lr_bits_init(tid);
  lr_stage(fp, g, cdef, dbk, src, U, tid);
  int w[6], ref[6];
#pragma unroll
  for (int k = 0; k < 6; k++) {
    w[k] = stats[u].w0[k];
    ref[k] = cs.ref[k];
  }
  LrTrace tr;
  lr_refine(fp.lambda, g, U, w, ref, &tr, tid);
  if (tid == 0) lr_record(stats[u], w, tr);
}
__global__ __launch_bounds__(LR_T) void k_lr_path(const Mav1FrameParams fp, const uint8_t *__restrict__ src,
                                                  const uint8_t *__restrict__ cdef, const uint8_t *__restrict__ dbk,
                                                  LrUnitStat *__restrict__ stats) {
  lr_path_body(fp, src, cdef, dbk, stats, blockIdx.x);
}

/* Per plane, units in raster order with the true running references: the
 * choice of lr_select (lr_search.c:262-349). LR_CB units at a time are scored
 * side by side under the running references, two per wave (lr_score), and
 * accepted up to the first that changes a reference or whose refinement has
 * to run again; that one and the next such units are then refined, one per
 * LR_T threads, and scored anew. After maxSteps such steps the launch records
 * where it stands and ends: references that change in a burst are followed
 * here, and where units keep coming out otherwise, k_lr_path refines all that
 * are left side by side under the reference then running, and the next launch
 * goes on. units[] and lrType[plane] receive the result, reruns[plane] the
 * number of refinements run here. The next units' statistics are loaded ahead.
 * Bound by the latency of a step, one per LR_CB units or change of a
 * reference, and by the refinements: 62 us for a 1920x1080 key frame, 240 us
 * with one thread accepting unit by unit in three launches. */
#define LR_CB 16
#define LR_CT 512 /* 32 threads per unit; the refinement takes about 200 registers */
#define LR_CG (LR_CT / LR_T)

/* The chain's staged units, their scores and choices. */
struct LrWalk {
  LrUnitStat st[LR_CB];
  Mav1LrUnit un[LR_CB];
  int tap[LR_CB][6];   /* the refined taps under the running reference */
  int flags[LR_CB];    /* 1: refine again, 2: changes a reference, 4: not NONE */
  int ref[6], refX[2]; /* running references */
  int next, nre, re[LR_CG], used;
  LrUnitLds re_[LR_CG];
};

/* 64-bit minimum over the lanes of a row of 16. */
DEVI unsigned long long lr_row_min(unsigned long long v) {
  auto step = [&](unsigned long long o) { v = o < v ? o : v; };
  step((unsigned long long)dpp_t64<DPP_QX1>((long long)v));
  step((unsigned long long)dpp_t64<DPP_QX2>((long long)v));
  step((unsigned long long)dpp_t64<DPP_HMIRROR>((long long)v));
  step((unsigned long long)dpp_t64<DPP_MIRROR>((long long)v));
  return v;
}

/* The choice of staged unit u (NONE, then WIENER, then the sets in order,
 * first strict minimum; the lr_test pattern) under the running references by
 * 32 lanes: one per self-guided set, then one per Wiener tap. odd: parity of
 * its index.
 * Each step of the refinement compares two costs that share the other taps'
 * bits. So every tap's step is decided anew from the record side by side,
 * and the record holds if all decide as recorded (the last may differ:
 * nothing follows it). */
DEVI void lr_score(int lambda, LrWalk &W, int p, int u, int odd, int lrTest, int lane) {
  const int l32 = lane & 31, set = lane & 15, k = set < 6 ? set : 5, j = k % 3, half = lane & 32;
  const bool tapLane = l32 >= 16 && set < 6 && j >= (p ? 1 : 0);
  const LrUnitStat &st = W.st[u];
  const int ref = W.ref[k], x0r = W.refX[0], x1r = W.refX[1];
  /* row 0: the sets */
  const int q0 = st.xqd[set][0], q1 = st.xqd[set][1];
  const uint32_t ss = st.sseSgr[set];
  int bits = 2 + SGRPROJ_PARAMS_BITS;
  if (SGR_PARAM(set, 0)) bits += lr_xqd_bits(0, x0r, q0);
  if (SGR_PARAM(set, 2)) bits += lr_xqd_bits(1, x1r, q1);
  const unsigned long long key =
      lr_row_min((unsigned long long)(lrTest ? (long long)ss : lr_rd(lambda, ss, bits)) << 4 | set);
  /* row 1: the taps */
  const int w0 = st.w0[k];
  const uint32_t cur = st.tr.cur[k], sm = st.tr.m[k], sp = st.tr.p[k];
  const int b1 = lr_tap_bits(j, ref, w0), bm = lr_tap_bits(j, ref, d_max(Wiener_Taps_Min[j], w0 - 1));
  const int bp = lr_tap_bits(j, ref, d_min(Wiener_Taps_Max[j], w0 + 1));
  const int d = lr_step(lambda, j, w0, cur, sm, sp, bm, b1, bp), tap = tapLane ? w0 + d : w0;
  const unsigned again = (unsigned)(__ballot(tapLane && k < 5 && tap != st.wStar[k]) >> half);
  const unsigned moved = (unsigned)(__ballot(tapLane && tap != ref) >> half);
  int wbits = tapLane ? (d < 0 ? bm : d > 0 ? bp : b1) : 0;
  wbits += dpp_t<DPP_QX1>(wbits);
  wbits += dpp_t<DPP_QX2>(wbits);
  wbits += dpp_t<DPP_HMIRROR>(wbits);
  wbits += dpp_t<DPP_MIRROR>(wbits);
  const long long wc = __shfl(lr_rd(lambda, d < 0 ? sm : d > 0 ? sp : cur, 2 + wbits), half + 21); /* the last tap's */
  const long long kmin = (long long)__shfl(key, half);
  const int bs = (int)(kmin & 15);
  long long best = lr_rd(lambda, st.sseNone, 1);
  int kind = RESTORE_NONE;
  if (wc < best) {
    best = wc;
    kind = RESTORE_WIENER;
  }
  if ((kmin >> 4) < best) kind = RESTORE_SGRPROJ;
  if (lrTest) kind = odd ? RESTORE_SGRPROJ : RESTORE_WIENER;
  const int n0 = st.xqd[bs][0], n1 = st.xqd[bs][1];
  Mav1LrUnit &un = W.un[u];
  if (l32 == 0) {
    const bool sg = kind == RESTORE_SGRPROJ;
    un.type = kind;
    un.set = sg ? bs : 0;
    un.xqd[0] = sg ? n0 : 0;
    un.xqd[1] = sg ? n1 : 0;
    W.flags[u] = (again ? 1 : 0) | ((kind == RESTORE_WIENER ? moved != 0 : sg && (n0 != x0r || n1 != x1r)) ? 2 : 0) |
                 (kind != RESTORE_NONE ? 4 : 0);
  }
  if (l32 >= 16 && set < 6) {
    un.wiener[k / 3][j] = kind == RESTORE_WIENER ? tap : 0;
    W.tap[u][k] = tap;
  }
}

/* After the scores of units li .. nb - 1: the references and the next unit
 * (first wave). */
DEVI void lr_accept(LrWalk &W, int p, int li, int nb, int lane) {
  const int f = li + lane < nb ? W.flags[li + lane] : 0;
  const unsigned long long again = __ballot(f & 1), stop = __ballot(f & 3);
  const int first = stop ? __ffsll((unsigned long long)stop) - 1 : nb - li; /* the first unit not followed by others */
  const bool re = (again >> (first & 63)) & (stop != 0);
  const int n = first + (stop && !re); /* units accepted */
  const unsigned long long used = __ballot((f & 4) && lane < n);
  if (stop && !re) {
    const Mav1LrUnit &un = W.un[li + first];
    if (un.type == RESTORE_WIENER && lane < 6 && lane % 3 >= (p ? 1 : 0)) W.ref[lane] = W.tap[li + first][lane];
    if (un.type == RESTORE_SGRPROJ && lane < 2) W.refX[lane] = un.xqd[lane];
  }
  /* the units to refine: the first one's place and the next like it */
  if (re && ((again >> lane) & 1)) {
    const int at = __popcll(again & ((1ull << lane) - 1));
    if (at < LR_CG) W.re[at] = li + lane;
  }
  if (lane == 0) {
    W.next = li + n;
    W.nre = re ? d_min(LR_CG, __popcll(again)) : 0;
    W.used |= used != 0;
  }
}

DEVI void lr_chain_body(const Mav1FrameParams &fp, const uint8_t *__restrict__ src, const uint8_t *__restrict__ cdef, const uint8_t *__restrict__ dbk, LrUnitStat *__restrict__ stats, Mav1LrUnit *__restrict__ units, int *__restrict__ lrType, int lrTest, int *__restrict__ reruns, int maxSteps, const int p) {
  const int tid = threadIdx.x;
  __shared__ LrWalk W;
  const int nu = fp.lr_unit_rows[p] * fp.lr_unit_cols[p], off = fp.lr_unit_off[p];
  LrChain &cs = stats[off].chain;
  if (cs.done) return;
  const int b00 = cs.start;
  constexpr int SW = (int)(sizeof(LrUnitStat) / 4), NV = (LR_CB * SW + LR_CT - 1) / LR_CT;
  int v[NV]; /* the next batch's statistics */
  auto fetch = [&](int b0) {
    const int words = d_min(LR_CB, nu - b0) * SW;
#pragma unroll
    for (int i = 0; i < NV; i++)
      if (tid + i * LR_CT < words) v[i] = ((const int *)(stats + off + b0))[tid + i * LR_CT];
  };
  lr_bits_init(tid);
  if (tid < 6) W.ref[tid] = cs.ref[tid];
  if (tid < 2) W.refX[tid] = cs.refX[tid];
  if (tid == 0) W.used = cs.used;
  for (int q = tid; q < LR_CB * (int)(sizeof(Mav1LrUnit) / 4); q += LR_CT) ((int *)W.un)[q] = 0; /* padding included */
  int nrerun = cs.nrerun, steps = 0;
  fetch(b00);
  for (int b0 = b00; b0 < nu; b0 += LR_CB) {
    const int nb = d_min(LR_CB, nu - b0);
#pragma unroll
    for (int i = 0; i < NV; i++)
      if (tid + i * LR_CT < nb * SW) ((int *)W.st)[tid + i * LR_CT] = v[i];
    if (b0 + LR_CB < nu) fetch(b0 + LR_CB);
    __syncthreads();
    int li = 0;
    bool stop = false;
    while (li < nb) {
      const int u = li + (tid >> 5);
      if (d_uni(tid >> 6) * 2 + li < nb) /* a wave's second unit may lie past the end: the last one once more */
        lr_score(fp.lambda, W, p, d_min(u, nb - 1), (b0 + d_min(u, nb - 1)) & 1, lrTest, tid & 63);
      __syncthreads();
      if (tid < 64) lr_accept(W, p, li, nb, tid);
      __syncthreads();
      li = W.next;
      const int nre = W.nre;
      if (!nre) continue;
      if (steps++ == maxSteps) {
        stop = true;
        break;
      }
      /* units again, under the running reference; then they are scored anew */
      const int grp = d_uni(tid / LR_T), t = tid % LR_T, ru = W.re[d_min(grp, nre - 1)];
      LrUnitLds &U = W.re_[grp];
      LrGeo g;
      lr_geo(fp, off + b0 + ru, g);
      lr_stage(fp, g, cdef, dbk, src, U, t);
      int w[6], ref[6];
#pragma unroll
      for (int k = 0; k < 6; k++) {
        w[k] = W.st[ru].w0[k];
        ref[k] = W.ref[k];
      }
      LrTrace tr;
      lr_refine(fp.lambda, g, U, w, ref, &tr, t);
      __syncthreads();
      if (t == 0 && grp < nre) lr_record(W.st[ru], w, tr);
      nrerun += nre;
      __syncthreads();
    }
    for (int q = tid; q < li * (int)(sizeof(Mav1LrUnit) / 4); q += LR_CT)
      ((int *)(units + off + b0))[q] = ((const int *)W.un)[q];
    if (stop) {
      if (tid == 0) {
        cs.start = b0 + li;
        cs.used = W.used;
        cs.nrerun = nrerun;
        for (int k = 0; k < 6; k++) cs.ref[k] = W.ref[k];
        for (int k = 0; k < 2; k++) cs.refX[k] = W.refX[k];
      }
      return;
    }
    __syncthreads();
  }
  if (tid == 0) {
    cs.done = 1;
    lrType[p] = W.used ? RESTORE_SWITCHABLE : RESTORE_NONE;
    reruns[p] = nrerun;
  }
}
__global__ __launch_bounds__(LR_CT) void k_lr_chain(const Mav1FrameParams fp, const uint8_t *__restrict__ src,
                                                    const uint8_t *__restrict__ cdef, const uint8_t *__restrict__ dbk,
                                                    LrUnitStat *__restrict__ stats, Mav1LrUnit *__restrict__ units,
                                                    int *__restrict__ lrType, int lrTest, int *__restrict__ reruns,
                                                    int maxSteps) {
  lr_chain_body(fp, src, cdef, dbk, stats, units, lrType, lrTest, reruns, maxSteps, blockIdx.x);
}

static_assert(sizeof(LrUnitStat) <= LR_STAT_MAX_BYTES, "LR_STAT_MAX_BYTES too small");
size_t lr_stat_bytes() { return sizeof(LrUnitStat); }

hipError_t launch_lr_fit(hipStream_t st, const Mav1FrameParams &fp, const uint8_t *src, const uint8_t *cdef,
                         const uint8_t *dbk, void *stats, int nunits) {
  hipLaunchKernelGGL(k_lr_fit, dim3(nunits, 3), dim3(LR_T), 0, st, fp, src, cdef, dbk, (LrUnitStat *)stats);
  return hipGetLastError();
}

/* Steps of a chain launch before the refinement pass. The number hardly
 * matters: 2, 4 and 8 took 575, 632 and 744 us where one reference holds for
 * most units, 4.98, 5.07 and 5.20 ms where it changes again and again
 * (1920x1080). */
#define LR_STEPS 4

hipError_t launch_lr_path(hipStream_t st, const Mav1FrameParams &fp, const uint8_t *src, const uint8_t *cdef,
                          const uint8_t *dbk, void *stats, int nunits) {
  hipLaunchKernelGGL(k_lr_path, dim3(nunits), dim3(LR_T), 0, st, fp, src, cdef, dbk, (LrUnitStat *)stats);
  return hipGetLastError();
}

hipError_t launch_lr_chain(hipStream_t st, const Mav1FrameParams &fp, const uint8_t *src, const uint8_t *cdef,
                           const uint8_t *dbk, void *stats, Mav1LrUnit *units, int *lrType, int lrTest, int *reruns,
                           int last) {
  hipLaunchKernelGGL(k_lr_chain, dim3(3), dim3(LR_CT), 0, st, fp, src, cdef, dbk, (LrUnitStat *)stats, units, lrType,
                     lrTest, reruns, last ? INT_MAX : LR_STEPS);
  return hipGetLastError();
}

/* ---- batched launches (batch.h): the same kernels over several frames ---- */

/* The fit over every frame's units: the workgroups in part-major order
 * (g.start over units; part = block / units), the long serial fits first, as
 * in the single-frame launch. */
__global__ __launch_bounds__(LR_T) void k_lr_fit_b(const BatchFrame *__restrict__ T, const BatchGrid g) {
  const int units = g.start[g.n], part = blockIdx.x / units;
  const BatchIdx b = batch_idx(g, blockIdx.x - part * units);
  const BatchFrame &F = T[b.f];
  lr_fit_body(F.fp, gptr(F.src), gptr(F.rec), gptr(F.dbk), (LrUnitStat *)gptr(F.lrstats), b.x, part);
}
__global__ __launch_bounds__(LR_CT) void k_lr_chain_b(const BatchFrame *__restrict__ T, int lrTest, int maxSteps) {
  const BatchFrame &F = T[blockIdx.x / 3];
  lr_chain_body(F.fp, gptr(F.src), gptr(F.rec), gptr(F.dbk), (LrUnitStat *)gptr(F.lrstats), gptr(F.lrunits),
                gptr(F.lrtype), lrTest, gptr(F.lrreruns), maxSteps, blockIdx.x % 3);
}

static BatchGrid unit_grid(const BatchFrame *H, int n) {
  BatchGrid g = batch_grid();
  for (int f = 0; f < n; f++) batch_grid_add(g, H[f].lr_units, 1, 1);
  return g;
}

hipError_t launch_lr_fit_b(hipStream_t st, const BatchFrame *T, const BatchFrame *H, int n) {
  const BatchGrid g = unit_grid(H, n);
  hipLaunchKernelGGL(k_lr_fit_b, dim3(g.start[n] * 3), dim3(LR_T), 0, st, T, g);
  return hipGetLastError();
}

__global__ __launch_bounds__(LR_T) void k_lr_path_b(const BatchFrame *__restrict__ T, const BatchGrid g) {
  const BatchIdx b = batch_idx(g);
  const BatchFrame &F = T[b.f];
  lr_path_body(F.fp, gptr(F.src), gptr(F.rec), gptr(F.dbk), (LrUnitStat *)gptr(F.lrstats), b.x);
}

hipError_t launch_lr_path_b(hipStream_t st, const BatchFrame *T, const BatchFrame *H, int n) {
  const BatchGrid g = unit_grid(H, n);
  hipLaunchKernelGGL(k_lr_path_b, dim3(g.start[n]), dim3(LR_T), 0, st, T, g);
  return hipGetLastError();
}

hipError_t launch_lr_chain_b(hipStream_t st, const BatchFrame *T, int n, int lrTest, int last) {
  hipLaunchKernelGGL(k_lr_chain_b, dim3(3 * n), dim3(LR_CT), 0, st, T, lrTest, last ? INT_MAX : LR_STEPS);
  return hipGetLastError();
}
