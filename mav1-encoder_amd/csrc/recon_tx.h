/* The transform stages of the reconstruction kernels (behaviour of
 * src/kernels/k_recon.h:39-173, k_fwd.h and k_itx.h) on the workgroup's LDS
 * gL, which the including file defines. */
#ifndef MAV1_RECON_TX_H
#define MAV1_RECON_TX_H

/* The lane index is opaque (d_local) so that the address arithmetic derived
 * from it stays inside each transform stage. */
DEVI TxCtx wg_ctx() {
  TxCtx c;
  c.tid = d_local(threadIdx.x);
  c.nt = RT;
  c.wg = true;
  c.red = gL.red;
  return c;
}
DEVI TxCtx wave_ctx() {
  TxCtx c;
  c.tid = d_local(threadIdx.x & 63);
  c.nt = 64;
  c.wg = false;
  c.red = nullptr;
  return c;
}
DEVI long long wg_sum64(long long v) { return tx_sum64(wg_ctx(), v); }
/* A workgroup barrier that orders LDS only: global stores before it (levels,
 * block records) need not have completed, as nothing in the workgroup reads
 * them back before the superblock is published with an agent-scope release. */
DEVI void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

/* ---- scan / tx-set helpers (spec 5.11.47 / 5.11.48) ---- */
DEVI const int16_t *scan_of(int txSz, int kind) {
  switch (txSz) {
    case TX_4X4: return kind == 1 ? Mrow_Scan_4x4 : kind == 2 ? Mcol_Scan_4x4 : Default_Scan_4x4;
    case TX_4X8: return kind == 1 ? Mrow_Scan_4x8 : kind == 2 ? Mcol_Scan_4x8 : Default_Scan_4x8;
    case TX_8X4: return kind == 1 ? Mrow_Scan_8x4 : kind == 2 ? Mcol_Scan_8x4 : Default_Scan_8x4;
    case TX_8X8: return kind == 1 ? Mrow_Scan_8x8 : kind == 2 ? Mcol_Scan_8x8 : Default_Scan_8x8;
    case TX_8X16: return kind == 1 ? Mrow_Scan_8x16 : kind == 2 ? Mcol_Scan_8x16 : Default_Scan_8x16;
    case TX_16X8: return kind == 1 ? Mrow_Scan_16x8 : kind == 2 ? Mcol_Scan_16x8 : Default_Scan_16x8;
    case TX_16X16: return kind == 1 ? Mrow_Scan_16x16 : kind == 2 ? Mcol_Scan_16x16 : Default_Scan_16x16;
    case TX_4X16: return kind == 1 ? Mrow_Scan_4x16 : kind == 2 ? Mcol_Scan_4x16 : Default_Scan_4x16;
    case TX_16X4: return kind == 1 ? Mrow_Scan_16x4 : kind == 2 ? Mcol_Scan_16x4 : Default_Scan_16x4;
    case TX_16X32: return Default_Scan_16x32;
    case TX_32X16: return Default_Scan_32x16;
    case TX_8X32: return Default_Scan_8x32;
    case TX_32X8: return Default_Scan_32x8;
    default: return Default_Scan_32x32;
  }
}
/* Offset of a transform size's scan among the staged small scans, -1 for
 * the 32- and 64-point sizes. */
DEVI int small_scan_off(int txSz) {
  switch (txSz) {
    case TX_4X4: return 0;
    case TX_8X8: return 16;
    case TX_16X16: return 80;
    case TX_4X8: return 336;
    case TX_8X4: return 368;
    case TX_8X16: return 400;
    case TX_16X8: return 528;
    case TX_4X16: return 656;
    case TX_16X4: return 720;
    default: return -1;
  }
}
DEVI int scan_kind(int t) {
  return (t == V_DCT || t == V_ADST || t == V_FLIPADST) ? 1 : (t == H_DCT || t == H_ADST || t == H_FLIPADST) ? 2 : 0;
}
DEVI const int16_t *get_scan(int txSz, int t) {
  if (txSz == TX_16X64) return Default_Scan_16x32;
  if (txSz == TX_64X16) return Default_Scan_32x16;
  if (Tx_Size_Sqr_Up[txSz] == TX_64X64) return Default_Scan_32x32;
  const int kind = scan_kind(t);
  const int off = small_scan_off(txSz);
  if (off >= 0) return gL.scans + kind * SCAN_SMALL + off;
  return scan_of(txSz, kind);
}
DEVI int get_tx_set(int txSz, int isInter, int reduced) {
  const int sq = Tx_Size_Sqr[txSz], up = Tx_Size_Sqr_Up[txSz];
  if (up > TX_32X32) return TX_SET_DCTONLY;
  if (isInter) return (reduced || up == TX_32X32) ? TX_SET_INTER_3 : sq == TX_16X16 ? TX_SET_INTER_2 : TX_SET_INTER_1;
  if (up == TX_32X32) return TX_SET_DCTONLY;
  return (reduced || sq == TX_16X16) ? TX_SET_INTRA_2 : TX_SET_INTRA_1;
}
DEVI int in_set(int set, int t, int isInter) { return isInter ? TX_IN_SET_INTER(set, t) : TX_IN_SET_INTRA(set, t); }
DEVI int seg_eob(int txSz) {
  if (txSz == TX_16X64 || txSz == TX_64X16) return 512;
  return d_min(1024, Tx_Width[txSz] * Tx_Height[txSz]);
}
DEVI int uv_tx_size(int bs) {
  const int t = Max_Tx_Size_Rect[SUBSAMPLED_SIZE(bs, 1, 1)];
  if (Tx_Width[t] == 64 || Tx_Height[t] == 64) return Tx_Width[t] == 16 ? TX_16X32 : Tx_Height[t] == 16 ? TX_32X16 : TX_32X32;
  return t;
}
DEVI int tile_start(const Mav1FrameParams &fp, int miCol) { return ((miCol >> 4) / fp.tile_w_sb) * fp.tile_w_sb * 16; }

/* find_eob (k_recon.h:50-54): 1 + last scan position with a non-zero level. */
DEVI int tx_eob(const TxCtx &c, const int32_t *q_, const int16_t *scan, int n) {
  const lds_i32 *q = lds(q_);
  if (!c.wg) {
    /* one wave: the last non-zero scan position from a ballot per 64
     * positions (no cross-lane reduction) */
    int e = 0;
    for (int k0 = 0; k0 < n; k0 += 64) {
      const int k = k0 + c.tid;
      const unsigned long long nz = __ballot(k < n && q[scan[k]] != 0);
      if (nz) e = k0 + 64 - __clzll(nz);
    }
    return e;
  }
  int m = 0;
  for (int k = c.tid; k < n; k += c.nt)
    if (q[scan[k]]) m = k + 1;
  return tx_max(c, m);
}
/* est_coef_bits (k_recon.h:39-48) */
DEVI int tx_bits(const TxCtx &c, const int32_t *q_, const int16_t *scan, int eob) {
  if (!eob) return 8;
  const lds_i32 *q = lds(q_);
  long long b = 0;
  for (int k = c.tid; k < eob; k += c.nt) {
    const int l = d_abs(q[scan[k]]);
    b += l ? 8 * (2 + 2 * d_floorlog2((unsigned)l)) : 6;
  }
  return 48 + 16 * d_floorlog2((unsigned)eob + 1) + (int)tx_sum64(c, b);
}

/* Residual of transform block (x, y), stored in the type's flipped order
 * (row strides: source SS, prediction S). */
DEVI void tx_residual(const TxCtx &c, const uint8_t *spx, int SS, const uint8_t *px, int S, int x, int y, int lw, int lh,
                      int t, int32_t *resid_, int rs) {
  lds_i32 *resid = lds(resid_);
  const int w = 1 << lw, h = 1 << lh, fud = flip_ud(t), flr = flip_lr(t);
  for (int k = c.tid; k < w * h; k += c.nt) {
    const int i = k >> lw, j = k & (w - 1);
    const int yy = y + (fud ? h - 1 - i : i), xx = x + (flr ? w - 1 - j : j);
    resid[i * rs + j] = (int)spx[yy * SS + xx] - (int)px[yy * S + xx];
  }
  tx_sync(c);
}
/* px += residual (inverse transform output in flipped order), clipped. */
DEVI void tx_add(const TxCtx &c, uint8_t *px, int S, int x, int y, int lw, int lh, int t, const int32_t *res_, int rs) {
  const lds_i32 *res = lds(res_);
  const int w = 1 << lw, h = 1 << lh, fud = flip_ud(t), flr = flip_lr(t);
  for (int k = c.tid; k < w * h; k += c.nt) {
    const int i = k >> lw, j = k & (w - 1);
    const int o = (y + (fud ? h - 1 - i : i)) * S + x + (flr ? w - 1 - j : j);
    px[o] = (uint8_t)d_clip1((int)px[o] + res[i * rs + j]);
  }
  tx_sync(c);
}

/* One candidate type of one transform block (k_recon.h:60-173 loop body):
 * levels into q, returns the eob; the RD cost 16 * SSE + lambda * bits / 8
 * in *costOut (0 when `direct`: a single type and no depth search). */
template <bool SMALL>
NOINL int tx_eval(const TxCtx &c, const Mav1FrameParams &fp, const uint8_t *__restrict__ spx, int SS, const uint8_t *px,
                  int S, int x, int y, int txSz, int plane, int t, bool direct, int32_t *resid, int rs, int32_t *tmp,
                  int32_t *coef, int32_t *q, int32_t *dq, int qs, const int32_t *__restrict__ mats,
                  long long *costOut) {
  /* one transform block per call: its size, plane, type and placement are
   * the same in every lane */
  txSz = d_uni(txSz);
  plane = d_uni(plane);
  t = d_uni(t);
  x = d_uni(x);
  y = d_uni(y);
  S = d_uni(S);
  SS = d_uni(SS);
  const int lw = d_uni(Tx_Width_Log2[txSz]), lh = d_uni(Tx_Height_Log2[txSz]), w = 1 << lw, h = 1 << lh;
  const int dcQ = fp.dc_q[plane], acQ = fp.ac_q[plane];
  tx_residual(c, spx, SS, px, S, x, y, lw, lh, t, resid, rs);
  /* transforms up to 16x16: the scans staged in LDS, addressed as LDS; the
   * one-wave path takes the eob from the quantiser (the largest inverse-scan
   * position of a non-zero level, plus one: tx_eob's value) */
  const int16_t *scan = SMALL ? gL.scans + scan_kind(t) * SCAN_SMALL + small_scan_off(txSz) : get_scan(txSz, t);
  int eob;
  if constexpr (SMALL) {
    eob = d_uni(tx_forward_quant_small(c, resid, rs, tmp, q, txSz, t, gL.smats, dcQ, acQ, gL.qrcp[plane][0],
                                       gL.qrcp[plane][1], gL.iscans + scan_kind(t) * SCAN_SMALL + small_scan_off(txSz)));
  } else {
    tx_forward<SMALL>(c, resid, rs, tmp, coef, txSz, t, mats, gL.smats);
    tx_quantize(c, coef, q, txSz, dcQ, acQ, gL.qrcp[plane][0], gL.qrcp[plane][1]);
    eob = d_uni(tx_eob(c, q, scan, d_uni(seg_eob(txSz))));
  }
  if (direct) {
    *costOut = 0;
    return eob;
  }
  long long e = 0;
  const lds_i32 *rl = lds(resid);
  if (eob > 0) {
    tx_dequant(c, q, dq, qs, txSz, dcQ, acQ);
    tx_inverse<SMALL>(c, dq, qs, resid, rs, txSz, t);
    const int fud = flip_ud(t), flr = flip_lr(t);
    for (int k = c.tid; k < w * h; k += c.nt) {
      const int i = k >> lw, j = k & (w - 1);
      const int yy = y + (fud ? h - 1 - i : i), xx = x + (flr ? w - 1 - j : j);
      const int d = (int)spx[yy * SS + xx] - d_clip1((int)px[yy * S + xx] + rl[i * rs + j]);
      e += d * d;
    }
  } else {
    for (int k = c.tid; k < w * h; k += c.nt) {
      const int v = rl[(k >> lw) * rs + (k & (w - 1))];
      e += v * v;
    }
  }
  const long long sse = tx_sum64(c, e);
  *costOut = sse * 16 + (long long)fp.lambda * tx_bits(c, q, scan, eob) / 8;
  return eob;
}

/* Lossless 4x4: forward WHT (k_fwd.h:112-136) and inverse WHT (7.13.2.10),
 * one thread. */
DEVI void wht_fwd(const int32_t *r, int32_t *out) {
  int t[16];
  for (int j = 0; j < 4; j++) {
    int a = r[j], b = r[4 + j], c = r[8 + j], d = r[12 + j];
    a += b;
    d -= c;
    int e = (a - d) >> 1;
    b = e - b;
    c = e - c;
    a -= c;
    d += b;
    t[j] = a;
    t[4 + j] = c;
    t[8 + j] = d;
    t[12 + j] = b;
  }
  for (int i = 0; i < 4; i++) {
    int a = t[4 * i], b = t[4 * i + 1], c = t[4 * i + 2], d = t[4 * i + 3];
    a += b;
    d -= c;
    int e = (a - d) >> 1;
    b = e - b;
    c = e - c;
    a -= c;
    d += b;
    out[4 * i] = a;
    out[4 * i + 1] = c;
    out[4 * i + 2] = d;
    out[4 * i + 3] = b;
  }
}
DEVI void wht_inv1(int32_t *T, int shift) {
  int32_t a = T[0] >> shift, c = T[1] >> shift, d = T[2] >> shift, b = T[3] >> shift;
  a += c;
  d -= b;
  int32_t e = (a - d) >> 1;
  b = e - b;
  c = e - c;
  a -= b;
  d += c;
  T[0] = a;
  T[1] = b;
  T[2] = c;
  T[3] = d;
}

/* One transform block whose prediction is in px (k_recon.h:60-173): the
 * cheapest of the candidate types (first minimum), its levels into coefOut,
 * its reconstruction into px. Returns the eob; the type and cost in
 * *outType / *outCost. */
NOINL int code_tx_block(const Mav1FrameParams &fp, const uint8_t *__restrict__ spx, uint8_t *px, int S, int x, int y,
                        int txSz, int plane, const int *cands, int nc, int32_t *coefOut,
                        const int32_t *__restrict__ mats, int *outType, long long *outCost) {
  RLds &L = gL;
  const int tid = threadIdx.x;
  const int lw = Tx_Width_Log2[txSz], lh = Tx_Height_Log2[txSz], w = 1 << lw, h = 1 << lh;
  const int tw = d_min(32, w), th = d_min(32, h);
  const int dcQ = fp.dc_q[plane], acQ = fp.ac_q[plane];
  if (fp.lossless) {
    if (tid == 0) {
      int32_t r16[16], q16[16];
      for (int i = 0; i < 4; i++)
        for (int j = 0; j < 4; j++) r16[i * 4 + j] = (int)spx[(y + i) * S + x + j] - (int)px[(y + i) * S + x + j];
      wht_fwd(r16, q16);
      int eob = 0;
      for (int c = 15; c >= 0; c--)
        if (q16[Default_Scan_4x4[c]]) {
          eob = c + 1;
          break;
        }
      for (int k = 0; k < 16; k++) coefOut[k] = q16[k];
      if (eob) {
        int32_t r4[16], T[4];
        for (int k = 0; k < 16; k++) {
          long long d = (long long)q16[k] * (k == 0 ? dcQ : acQ), ad = d < 0 ? -d : d;
          long long d2 = ad & 0xFFFFFF;
          r4[k] = d_clip(-(1 << 15), (1 << 15) - 1, (int)(d < 0 ? -d2 : d2));
        }
        for (int i = 0; i < 4; i++) {
          for (int j = 0; j < 4; j++) T[j] = r4[i * 4 + j];
          wht_inv1(T, 2);
          for (int j = 0; j < 4; j++) r4[i * 4 + j] = d_clip(-(1 << 15), (1 << 15) - 1, T[j]);
        }
        for (int j = 0; j < 4; j++) {
          for (int i = 0; i < 4; i++) T[i] = r4[i * 4 + j];
          wht_inv1(T, 0);
          for (int i = 0; i < 4; i++) r4[i * 4 + j] = T[i];
        }
        for (int i = 0; i < 4; i++)
          for (int j = 0; j < 4; j++) {
            const int o = (y + i) * S + x + j;
            px[o] = (uint8_t)d_clip1((int)px[o] + r4[i * 4 + j]);
          }
      }
      L.ival[0] = eob;
    }
    __syncthreads();
    const int eob = L.ival[0];
    __syncthreads();
    *outType = DCT_DCT;
    *outCost = 0;
    return eob;
  }
  const bool direct = nc == 1 && !fp.tx_mode_select;
  /* up to 16x16: one candidate per wave; larger: the whole workgroup per
   * candidate. One code path for both keeps a single inlined copy of the
   * transform stages. */
  const bool small = w <= 16 && h <= 16;
  const int wave = tid >> 6, per = small ? RW : 1;
  const TxCtx c = small ? wave_ctx() : wg_ctx();
  int32_t *resid, *tmp, *coef, *qtry, *dq, *qbest;
  int rs, qs;
  if (small) {
    SmallTx &W = L.u.sm[wave];
    resid = W.resid, tmp = W.tmp, coef = W.coef, qtry = W.q, dq = W.dq, qbest = L.qbest, rs = SRS, qs = SQS;
  } else {
    BigTx &B = L.u.big;
    resid = B.resid, tmp = B.tmp, coef = B.coef, qtry = B.qtry, dq = B.dq, qbest = B.qbest, rs = BRS, qs = BQS;
  }
  long long bestCost = -1;
  int bestType = DCT_DCT, bestEob = 0;
  /* the candidates read the block's source and prediction from LDS */
  for (int k = tid; k < w * h; k += RT) {
    const int o = (y + (k >> lw)) * S + x + (k & (w - 1));
    L.tsrc[k] = spx[o];
    L.tpred[k] = px[o];
  }
  __syncthreads();
  for (int r0 = 0; r0 < nc; r0 += per) {
    const int ci = r0 + (small ? wave : 0);
    if (ci < nc) {
      long long cost;
      const int eob = tx_eval<false>(c, fp, L.tsrc, w, L.tpred, w, 0, 0, txSz, plane, cands[ci], direct, resid, rs, tmp, coef,
                              qtry, dq, qs, mats, &cost);
      if (c.tid == 0) {
        L.candCost[ci] = cost;
        L.candEob[ci] = eob;
      }
    }
    __syncthreads();
    /* first minimum in candidate order */
    int pick = -1;
    for (int k = r0; k < d_min(nc, r0 + per); k++)
      if (bestCost < 0 || L.candCost[k] < bestCost) {
        bestCost = L.candCost[k];
        pick = k;
      }
    if (pick >= 0) {
      bestEob = L.candEob[pick];
      bestType = bestEob > 0 ? cands[pick] : DCT_DCT;
      const int32_t *from = small ? L.u.sm[pick - r0].q : L.u.big.qtry;
      for (int k = tid; k < tw * th; k += RT) qbest[k] = from[k];
    }
    __syncthreads();
  }
  for (int k = tid; k < tw * th; k += RT) coefOut[k] = qbest[k];
  if (bestEob > 0 && (!small || wave == 0)) {
    tx_dequant(c, qbest, dq, qs, txSz, dcQ, acQ);
    tx_inverse(c, dq, qs, resid, rs, txSz, bestType);
    tx_add(c, px, S, x, y, lw, lh, bestType, resid, rs);
  }
  __syncthreads();
  *outType = bestType;
  *outCost = bestCost;
  return bestEob;
}

/* The workgroup's constant tables in LDS: the short forward matrices, the
 * small transforms' scans and the quantiser reciprocals. */
DEVI void stage_smats(const Mav1FrameParams &fp, const int32_t *__restrict__ mats) {
  for (int q = threadIdx.x; q < TX_SMATS; q += RT) {
    const int kind = q / 336, r = q - kind * 336;
    const int n = r < 16 ? 2 : r < 80 ? 3 : 4, idx = r - (n == 2 ? 0 : n == 3 ? 16 : 80);
    gL.smats[q] = mats[(kind * 5 + n - 2) * 4096 + idx];
  }
  const int sizes[9] = {TX_4X4, TX_8X8, TX_16X16, TX_4X8, TX_8X4, TX_8X16, TX_16X8, TX_4X16, TX_16X4};
  for (int q = threadIdx.x; q < 3 * SCAN_SMALL; q += RT) {
    const int kind = q / SCAN_SMALL, r = q - kind * SCAN_SMALL;
    int k = 8;
    while (small_scan_off(sizes[k]) > r) k--;
    const int off = small_scan_off(sizes[k]), v = scan_of(sizes[k], kind)[r - off];
    gL.scans[q] = v;
    gL.iscans[kind * SCAN_SMALL + off + v] = r - off;
  }
  if (threadIdx.x < 6) {
    const int p = threadIdx.x >> 1;
    gL.qrcp[p][threadIdx.x & 1] = tx_qrcp((threadIdx.x & 1) ? fp.ac_q[p] : fp.dc_q[p]);
  }
}

#endif
