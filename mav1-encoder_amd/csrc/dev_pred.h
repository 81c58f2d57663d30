/* Prediction helpers for the analysis and reconstruction kernels: unscaled
 * inter prediction (AV1 spec 7.11.3.3-7.11.3.4) of 4x4 units in registers from
 * an LDS-staged reference window, intra edge preparation (7.11.2 steps 1-3),
 * the intra predictor per sample and per 4x4 unit, and 4x4 Hadamard SATD.
 * Functions with a template argument NT are called by every thread of a
 * workgroup of NT threads (a wave64 by default); `lane` is the thread's index
 * in the workgroup. */
#ifndef MAV1_DEV_PRED_H
#define MAV1_DEV_PRED_H

#include "dev_common.h"

/* Sum over the NT threads of the workgroup; every thread gets it. Beyond
 * one wave, the waves' sums meet in LDS between two barriers (the first
 * keeps a previous sum's readers ahead of the writes). */
template <int NT>
DEVI int group_sum(int v) {
  v = wave_sum_dpp(v);
  if constexpr (NT == 64) {
    return v;
  } else {
    __shared__ int part[NT / 64];
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; i++) t += part[i];
    return t;
  }
}

/* ---- inter ---- */
typedef __attribute__((address_space(3))) const uint32_t lds_word;
/* A plane's prediction from one reference (7.11.3.3-7.11.3.4, EIGHTTAP, or
 * its 4-tap form for blocks of 4): the window's first sample in the plane,
 * and the taps: horizontal ones as signed bytes for the dot products with
 * (sample - 128) (a whole-sample phase's 128 as 2 * 64, hs = 1), vertical
 * ones as pairs of 16 bits. */
struct InterTaps {
  uint32_t h[2], v[4];
  int hs, y0, x0;
};
DEVI void inter_taps(InterTaps &T, int x, int y, int w, int h, int mvr, int mvc, int sub) {
  const int posX = ((x << SUBPEL_BITS) + ((2 * mvc) >> sub)) * 64 + 32;
  const int posY = ((y << SUBPEL_BITS) + ((2 * mvr) >> sub)) * 64 + 32;
  const int px = (posX >> 6) & SUBPEL_MASK, py = (posY >> 6) & SUBPEL_MASK;
  const int16_t *th = SUBPEL_FILTER(w <= 4 ? 4 : EIGHTTAP, px), *tv = SUBPEL_FILTER(h <= 4 ? 4 : EIGHTTAP, py);
  uint32_t a[2] = {0, 0};
#pragma unroll
  for (int t = 0; t < 8; t++) {
    a[t >> 2] |= (uint32_t)((px ? th[t] : th[t] / 2) & 255) << (8 * (t & 3));
    if (!(t & 1)) T.v[t >> 1] = (uint32_t)(tv[t] & 0xFFFF) | (uint32_t)(tv[t + 1] & 0xFFFF) << 16;
  }
  T.h[0] = a[0];
  T.h[1] = a[1];
  T.hs = px ? 0 : 1;
  T.y0 = (posY >> 10) - 3;
  T.x0 = (posX >> 10) - 3;
}
/* The reference samples a w x h block's prediction reads, coordinates
 * clamped, into win (row stride ws). */
template <int NT>
DEVI void inter_stage(const uint8_t *__restrict__ plane, int S, int lastX, int lastY, const InterTaps &T, int w, int h,
                      uint8_t *win, int ws, int lane) {
  const int n = w + 7, M = ((1 << 20) + n - 1) / n; /* k / n for k < 71 * 71 */
  for (int k = lane; k < n * (h + 7); k += NT) {
    const int r = (k * M) >> 20, c = k - r * n;
    win[r * ws + c] = plane[d_clip(0, lastY, T.y0 + r) * S + d_clip(0, lastX, T.x0 + c)];
  }
}
/* The prediction of the 4x4 unit at window position `at` (eight-tap support
 * included), a row per word. */
DEVI void inter_unit(const InterTaps &T, const uint8_t *win, int ws, int at, uint32_t out[4]) {
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  union P {
    uint32_t u;
    s16x2 v;
  };
  const int t0 = (int)T.h[0], t1 = (int)T.h[1], sh = T.hs;
  const int s = at & 3;
  int m[4][11];
#pragma unroll
  for (int r = 0; r < 11; r++) {
    const lds_word *q = (const lds_word *)(win + (at & ~3) + r * ws);
    const uint32_t q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
    const uint32_t n0 = __builtin_amdgcn_alignbyte(q1, q0, s) ^ 0x80808080u;
    const uint32_t n1 = __builtin_amdgcn_alignbyte(q2, q1, s) ^ 0x80808080u;
    const uint32_t n2 = __builtin_amdgcn_alignbyte(q3, q2, s) ^ 0x80808080u;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int lo = (int)__builtin_amdgcn_alignbyte(n1, n0, j), hi = (int)__builtin_amdgcn_alignbyte(n2, n1, j);
      const int a = __builtin_amdgcn_sdot4(hi, t1, __builtin_amdgcn_sdot4(lo, t0, 0, false), false);
      m[j][r] = ((a << sh) + 16384 + 4) >> 3;
    }
  }
  P v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    v[i].u = T.v[i];
    out[i] = 0;
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    P p[10];
#pragma unroll
    for (int r = 0; r < 10; r++) p[r].u = ((uint32_t)m[j][r] & 0xFFFF) | (uint32_t)m[j][r + 1] << 16;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      int a = 1 << 10;
#pragma unroll
      for (int t = 0; t < 4; t++) a = __builtin_amdgcn_sdot2(p[i + 2 * t].v, v[t].v, a, false);
      out[i] |= (uint32_t)d_clip1(a >> 11) << (8 * j);
    }
  }
}
/* SATD of a 4x4 unit, rows as words. */
DEVI int unit_satd(const uint32_t s[4], const uint32_t p[4]) {
  int d[16];
#pragma unroll
  for (int k = 0; k < 16; k++) d[k] = (int)((s[k >> 2] >> (8 * (k & 3))) & 255) - (int)((p[k >> 2] >> (8 * (k & 3))) & 255);
  return satd4x4_arr(d);
}
DEVI void unit_load(const uint8_t *s, int st, uint32_t out[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++) out[i] = *(const lds_word *)(s + i * st);
}
/* (a + b + 1) >> 1 of four samples */
DEVI uint32_t avg4(uint32_t a, uint32_t b) { return (a | b) - (((a ^ b) >> 1) & 0x7F7F7F7Fu); }

/* ---- intra ---- */
#define EDGE_NEG 16 /* edge arrays are addressed from index -EDGE_NEG */

/* Neighbouring samples (7.11.2 steps 1-3) of a w x h block at plane (x, y):
 * A[0 .. w+h-1] above, L[0 .. w+h-1] left, A[-1] = L[-1] = the corner. */
template <int NT = 64>
DEVI void wave_intra_edges(const uint8_t *px, int S, int x, int y, int w, int h, int hl, int ha, int har, int hbl,
                           int maxX, int maxY, int *A, int *L, int lane) {
  const int aLim = d_min(maxX, x + (har ? 2 * w : w) - 1), lLim = d_min(maxY, y + (hbl ? 2 * h : h) - 1);
  for (int i = lane; i < w + h; i += NT) {
    A[i] = ha ? px[(y - 1) * S + d_min(aLim, x + i)] : hl ? px[y * S + x - 1] : 127;
    L[i] = hl ? px[d_min(lLim, y + i) * S + x - 1] : ha ? px[(y - 1) * S + x] : 129;
  }
  if (lane == 0) {
    int corner = (ha && hl) ? px[(y - 1) * S + x - 1] : ha ? px[(y - 1) * S + x] : hl ? px[y * S + x - 1] : 128;
    A[-1] = L[-1] = corner;
  }
  __syncthreads();
}

DEVI const uint8_t *sm_weights(int lg) {
  return lg == 2 ? Sm_Weights_Tx_4x4 : lg == 3 ? Sm_Weights_Tx_8x8 : lg == 4 ? Sm_Weights_Tx_16x16
         : lg == 5 ? Sm_Weights_Tx_32x32 : Sm_Weights_Tx_64x64;
}

/* Per-block constants of one intra mode. */
struct IntraMode {
  int mode, pAngle, dx, dy, upA, upL, dcv, lw, lh, corner;
};

DEVI void intra_mode_setup(IntraMode &m, int mode, int delta, int lw, int lh) {
  m.mode = mode;
  m.lw = lw;
  m.lh = lh;
  m.upA = m.upL = 0;
  m.dx = m.dy = 0;
  m.pAngle = 0;
  if (mode >= V_PRED && mode <= D67_PRED) {
    int pa = Mode_To_Angle[mode] + delta * ANGLE_STEP;
    m.pAngle = pa;
    if (pa < 90) m.dx = Dr_Intra_Derivative[pa];
    else if (pa > 90 && pa < 180) m.dx = Dr_Intra_Derivative[180 - pa];
    if (pa > 90 && pa < 180) m.dy = Dr_Intra_Derivative[pa - 90];
    else if (pa > 180) m.dy = Dr_Intra_Derivative[270 - pa];
  }
}

/* DC value (7.11.2.5 DC_PRED) from the edges; every lane gets it. */
template <int NT = 64>
DEVI int wave_intra_dc(const int *A, const int *L, int w, int h, int lw, int lh, int hl, int ha, int lane) {
  int s = 0;
  for (int i = lane; i < w; i += NT) s += ha ? A[i] : 0;
  for (int i = lane; i < h; i += NT) s += hl ? L[i] : 0;
  s = group_sum<NT>(s);
  if (ha && hl) return (s + ((w + h) >> 1)) / (w + h);
  if (hl) return d_clip1((s + (h >> 1)) >> lh);
  if (ha) return d_clip1((s + (w >> 1)) >> lw);
  return 128;
}

/* Predicted sample (i, j) of the block (7.11.2.4 - 7.11.2.7). */
DEVI int intra_px(const IntraMode &m, const int *A, const int *L, int i, int j) {
  const int w = 1 << m.lw, h = 1 << m.lh;
  switch (m.mode) {
    case DC_PRED: return m.dcv;
    case SMOOTH_PRED: {
      const uint8_t *wx = sm_weights(m.lw), *wy = sm_weights(m.lh);
      return d_round2(wy[i] * A[j] + (256 - wy[i]) * L[h - 1] + wx[j] * L[i] + (256 - wx[j]) * A[w - 1], 9);
    }
    case SMOOTH_V_PRED: {
      const uint8_t *wy = sm_weights(m.lh);
      return d_round2(wy[i] * A[j] + (256 - wy[i]) * L[h - 1], 8);
    }
    case SMOOTH_H_PRED: {
      const uint8_t *wx = sm_weights(m.lw);
      return d_round2(wx[j] * L[i] + (256 - wx[j]) * A[w - 1], 8);
    }
    case PAETH_PRED: {
      int base = A[j] + L[i] - m.corner;
      int pl = d_abs(base - L[i]), pt = d_abs(base - A[j]), ptl = d_abs(base - m.corner);
      return (pl <= pt && pl <= ptl) ? L[i] : pt <= ptl ? A[j] : m.corner;
    }
    default: break;
  }
  const int pa = m.pAngle, upA = m.upA, upL = m.upL;
  if (pa == 90) return A[j];
  if (pa == 180) return L[i];
  if (pa < 90) {
    int idx = (i + 1) * m.dx, base = (idx >> (6 - upA)) + (j << upA), sh = ((idx * (1 << upA)) >> 1) & 31;
    int maxBase = (w + h - 1) << upA;
    return base < maxBase ? d_round2(A[base] * (32 - sh) + A[base + 1] * sh, 5) : A[maxBase];
  }
  if (pa < 180) {
    int idx = (j << 6) - (i + 1) * m.dx, base = idx >> (6 - upA);
    if (base >= -(1 << upA)) {
      int sh = ((idx * (1 << upA)) >> 1) & 31;
      return d_round2(A[base] * (32 - sh) + A[base + 1] * sh, 5);
    }
    idx = (i << 6) - (j + 1) * m.dy;
    base = idx >> (6 - upL);
    int sh = ((idx * (1 << upL)) >> 1) & 31;
    return d_round2(L[base] * (32 - sh) + L[base + 1] * sh, 5);
  }
  int idx = (j + 1) * m.dy, base = (idx >> (6 - upL)) + (i << upL), sh = ((idx * (1 << upL)) >> 1) & 31;
  return d_round2(L[base] * (32 - sh) + L[base + 1] * sh, 5);
}

/* Predicted samples of the 4x4 unit (uy, ux) of the block (7.11.2.4 -
 * 7.11.2.7). The mode may differ between lanes: each mode's samples are made
 * together. */
DEVI void intra_unit(const IntraMode &m, const int *A, const int *L, int uy, int ux, int p[16]) {
  const int w = 1 << m.lw, h = 1 << m.lh, i0 = uy * 4, j0 = ux * 4;
#define UNIT_LOOP _Pragma("unroll") for (int k = 0; k < 16; k++)
  const bool smooth = m.mode == SMOOTH_PRED || m.mode == SMOOTH_V_PRED || m.mode == SMOOTH_H_PRED;
  if (m.mode == DC_PRED) {
    UNIT_LOOP p[k] = m.dcv;
  } else if (smooth || m.mode == PAETH_PRED || m.pAngle == 90 || m.pAngle == 180) {
    /* modes of the row's left and the column's above sample */
    int a[4], l[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      a[t] = A[j0 + t];
      l[t] = L[i0 + t];
    }
    if (smooth) {
      const uint8_t *wx = sm_weights(m.lw) + j0, *wy = sm_weights(m.lh) + i0;
      const int bl = L[h - 1], ar = A[w - 1];
      /* weights in 256ths of the vertical and horizontal interpolation: the
       * one-directional modes leave the other out */
      const int v = m.mode != SMOOTH_H_PRED, hz = m.mode != SMOOTH_V_PRED, n = v + hz + 7;
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int gy = wy[t], gx = wx[u];
          const int sv = gy * a[u] + (256 - gy) * bl, sh = gx * l[t] + (256 - gx) * ar;
          p[4 * t + u] = ((v ? sv : 0) + (hz ? sh : 0) + (1 << (n - 1))) >> n;
        }
    } else if (m.mode == PAETH_PRED) {
      UNIT_LOOP {
        const int t = a[k & 3], q = l[k >> 2], base = t + q - m.corner;
        const int pl = d_abs(base - q), pt = d_abs(base - t), ptl = d_abs(base - m.corner);
        p[k] = (pl <= pt && pl <= ptl) ? q : pt <= ptl ? t : m.corner;
      }
    } else {
      const bool up = m.pAngle == 90;
      UNIT_LOOP p[k] = up ? a[k & 3] : l[k >> 2];
    }
  } else if (m.pAngle < 90) {
    const int maxBase = (w + h - 1) << m.upA;
    UNIT_LOOP {
      const int i = i0 + (k >> 2), j = j0 + (k & 3);
      const int idx = (i + 1) * m.dx, base = (idx >> (6 - m.upA)) + (j << m.upA), sh = ((idx * (1 << m.upA)) >> 1) & 31;
      const int b = d_min(base, maxBase), v = d_round2(A[b] * (32 - sh) + A[d_min(base + 1, maxBase)] * sh, 5);
      p[k] = base < maxBase ? v : A[maxBase];
    }
  } else if (m.pAngle < 180) {
    UNIT_LOOP {
      const int i = i0 + (k >> 2), j = j0 + (k & 3);
      const int ia = (j << 6) - (i + 1) * m.dx, ba = ia >> (6 - m.upA);
      const int il = (i << 6) - (j + 1) * m.dy, bl = il >> (6 - m.upL);
      const bool up = ba >= -(1 << m.upA);
      const int *E = up ? A : L;
      const int base = up ? ba : bl, sh = ((up ? ia * (1 << m.upA) : il * (1 << m.upL)) >> 1) & 31;
      p[k] = d_round2(E[base] * (32 - sh) + E[base + 1] * sh, 5);
    }
  } else {
    UNIT_LOOP {
      const int i = i0 + (k >> 2), j = j0 + (k & 3);
      const int idx = (j + 1) * m.dy, base = (idx >> (6 - m.upL)) + (i << m.upL), sh = ((idx * (1 << m.upL)) >> 1) & 31;
      p[k] = d_round2(L[base] * (32 - sh) + L[base + 1] * sh, 5);
    }
  }
#undef UNIT_LOOP
}

#endif
