/* Closed-loop reconstruction on gfx950 (behaviour of src/kernels/k_recon.h:
 * recon_sb / recon_block / code_plane / code_tx_block, in decode order, with
 * the dependencies of src/backend_cpu.c:81-86) and the intra edge filter
 * types of the frame driver (src/encoder.c:319-346).
 *
 * Inter blocks never read reconstructed neighbours: k_recon_list gathers
 * every inter block of the frame into a work list, and the persistent
 * 512-thread workgroups of k_recon_inter take blocks off it with an atomic
 * counter. Intra blocks read the reconstruction of earlier blocks: the
 * intra phase is one dataflow launch. k_intra_sched lists the superblocks
 * holding intra blocks in an order where every neighbour a superblock reads
 * (left, above-left, above, above-right within its tile column) comes
 * first; the persistent workgroups of k_recon_intra (recon_intra.h) take
 * list entries and wait (bounded, with an error word) for the done flags of
 * those neighbours.
 *
 * Inside a workgroup the candidates of every search run side by side: the
 * transform types of a block of at most 16x16 one per wave (each wave codes
 * its candidate alone: residual, forward transform, quantiser, eob and
 * rate, inverse transform and distortion), the nine dual-filter pairs over
 * three shared horizontal passes. Larger transforms (32- and 64-point) use
 * the whole workgroup per candidate. */
#include "recon_lds.h"
#include "recon_queue.h"

/* Inter prediction: the reference window and the horizontal pass of up to
 * three filters; compound: the first prediction and a band of the second. */
struct PredLds {
  uint8_t win[71 * 72];
  int16_t mid[3][71 * 64];
};
struct CompLds {
  uint8_t win[71 * 72];
  int16_t mid[71 * 64];
  int32_t p0[64 * 64];
  int32_t p1[16 * 64];
};

/* The working set of the workgroup that reconstructs an inter block. */
struct RLds : RCommon {
  union {
    SmallTx sm[RW];
    BigTx big;
    PredLds pr;
    CompLds cp;
  } u;
  long long fcost[9];
};
__shared__ RLds gL;

#include "recon_tx.h"

/* ---- inter prediction by the workgroup ---- */
DEVI void filter_taps(int w, int h, int filter, int posX, int posY, int *kh, int *kv) {
  int fv = filter & 3, fh = (filter >> 2) & 3;
  if (w <= 4) fh = (fh == EIGHTTAP_SMOOTH) ? 5 : (fh == EIGHTTAP || fh == EIGHTTAP_SHARP) ? 4 : fh;
  if (h <= 4) fv = (fv == EIGHTTAP_SMOOTH) ? 5 : (fv == EIGHTTAP || fv == EIGHTTAP_SHARP) ? 4 : fv;
  const int16_t *th = SUBPEL_FILTER(fh, (posX >> 6) & SUBPEL_MASK), *tv = SUBPEL_FILTER(fv, (posY >> 6) & SUBPEL_MASK);
#pragma unroll
  for (int t = 0; t < 8; t++) {
    kh[t] = th[t];
    kv[t] = tv[t];
  }
}
/* The (h + 7) x (w + 7) reference samples of the block (row stride w + 8),
 * clamped to the reference plane (7.11.3.3). */
DEVI void load_window(const uint8_t *__restrict__ plane, int S, int refW, int refH, int ix, int iy, int w, int h, int sub,
                      uint8_t *win, int tid) {
  const int lastX = ((refW + sub) >> sub) - 1, lastY = ((refH + sub) >> sub) - 1;
  const int WW = w + 8, nr = h + 7;
  for (int k = tid; k < nr * (w + 7); k += RT) {
    const int r = k / (w + 7), c = k - r * (w + 7);
    win[r * WW + c] = plane[d_clip(0, lastY, iy - 3 + r) * S + d_clip(0, lastX, ix - 3 + c)];
  }
}
DEVI void hpass(const uint8_t *win, int w, int h, const int *kh, int16_t *mid, int tid) {
  const int WW = w + 8;
  for (int k = tid; k < (h + 7) * w; k += RT) {
    const int r = k / w, c = k - r * w;
    const uint8_t *q = win + r * WW + c;
    int acc = 0;
#pragma unroll
    for (int t = 0; t < 8; t++) acc += kh[t] * q[t];
    mid[k] = (int16_t)d_round2(acc, 3);
  }
}

/* Inter prediction of a w x h block of one plane (7.11.3): round1 11 writes
 * clipped bytes to dst (row stride ds), round1 7 (compound) the unclipped
 * int32 values to dst32. */
NOINL void predict_inter_plane(const uint8_t *__restrict__ plane, int S, int refW, int refH, int x, int y, int w, int h,
                               int mvr, int mvc, int sub, int filter, uint8_t *dst, int ds, int32_t *dst32, int round1,
                               uint8_t *win, int16_t *mid) {
  const int tid = threadIdx.x;
  const int posX = ((x << SUBPEL_BITS) + ((2 * mvc) >> sub)) * 64 + 32;
  const int posY = ((y << SUBPEL_BITS) + ((2 * mvr) >> sub)) * 64 + 32;
  int kh[8], kv[8];
  filter_taps(w, h, filter, posX, posY, kh, kv);
  load_window(plane, S, refW, refH, posX >> 10, posY >> 10, w, h, sub, win, tid);
  __syncthreads();
  hpass(win, w, h, kh, mid, tid);
  __syncthreads();
  for (int k = tid; k < h * w; k += RT) {
    const int r = k / w, c = k - r * w;
    int acc = 0;
#pragma unroll
    for (int t = 0; t < 8; t++) acc += kv[t] * mid[(r + t) * w + c];
    if (round1 == 11) dst[r * ds + c] = (uint8_t)d_clip1(d_round2(acc, 11));
    else dst32[r * ds + c] = d_round2(acc, round1);
  }
  __syncthreads();
}

/* The dual-filter choice of a single-reference inter block (k_recon.h:
 * 312-334): SSE of the luma prediction of each of the 9 filter pairs over
 * the visible area, + lambda per non-regular filter, first minimum. The
 * window is shared, the three horizontal passes are computed once, each
 * wave scores pairs. */
NOINL int dual_filter_search(const Mav1FrameParams &fp, const uint8_t *__restrict__ refp,
                             const uint8_t *__restrict__ src) {
  RLds &L = gL;
  const Mav1BlockInfo &b = L.blk;
  const int tid = threadIdx.x, bs = b.bsize;
  const int w = BLOCK_WIDTH(bs), h = BLOCK_HEIGHT(bs), x0 = b.mi_col * 4, y0 = b.mi_row * 4, S = fp.stride[0];
  const int vw = d_min(w, fp.frame_w - x0), vh = d_min(h, fp.frame_h - y0);
  const int posX = ((x0 << SUBPEL_BITS) + 2 * b.mv_col) * 64 + 32, posY = ((y0 << SUBPEL_BITS) + 2 * b.mv_row) * 64 + 32;
  load_window(refp + fp.offset[0], S, fp.frame_w, fp.frame_h, posX >> 10, posY >> 10, w, h, 0, L.u.pr.win, tid);
  __syncthreads();
  for (int f = 0; f < 3; f++) {
    int kh[8], kv[8];
    filter_taps(w, h, f << 2, posX, posY, kh, kv);
    hpass(L.u.pr.win, w, h, kh, L.u.pr.mid[f], tid);
  }
  __syncthreads();
  const int wave = tid >> 6, lane = tid & 63;
  const uint8_t *sp = src + fp.offset[0] + y0 * S + x0;
  for (int f = wave; f < 9; f += RW) {
    int kh[8], kv[8];
    filter_taps(w, h, f % 3, posX, posY, kh, kv);
    const int16_t *mid = L.u.pr.mid[f / 3];
    long long e = 0;
    for (int k = lane; k < vw * vh; k += 64) {
      const int r = k / vw, c = k - r * vw;
      int acc = 0;
#pragma unroll
      for (int t = 0; t < 8; t++) acc += kv[t] * mid[(r + t) * w + c];
      const int d = d_clip1(d_round2(acc, 11)) - (int)sp[r * S + c];
      e += d * d;
    }
    e = wave_sum64(e);
    if (lane == 0) L.fcost[f] = e * 16 + (long long)fp.lambda * ((f % 3 != 0) + (f / 3 != 0));
  }
  __syncthreads();
  long long best = -1;
  int bestF = 0;
  for (int f = 0; f < 9; f++)
    if (best < 0 || L.fcost[f] < best) {
      best = L.fcost[f];
      bestF = (f % 3) | ((f / 3) << 2);
    }
  __syncthreads();
  return bestF;
}

/* code_plane (k_recon.h:190-291) for the inter block in L.blk, whose
 * prediction is in the frame rec. */
NOINL void code_inter_plane(const Mav1FrameParams &fp, const uint8_t *__restrict__ src, uint8_t *rec,
                            int32_t *__restrict__ coefs, const int32_t *__restrict__ mats, int plane, int txSz) {
  RLds &L = gL;
  Mav1BlockInfo &b = L.blk;
  const int tid = threadIdx.x;
  const int bs = b.bsize, sub = plane > 0, S = fp.stride[plane];
  const int psz = SUBSAMPLED_SIZE(bs, sub, sub);
  const int n4w = Num_4x4_Blocks_Wide[psz], n4h = Num_4x4_Blocks_High[psz];
  const int baseX = (b.mi_col >> sub) * 4, baseY = (b.mi_row >> sub) * 4;
  uint8_t *px = rec + fp.offset[plane];
  const uint8_t *spx = src + fp.offset[plane];
  const int stepX = Tx_Width[txSz] >> 2, stepY = Tx_Height[txSz] >> 2;
  const int set = get_tx_set(txSz, 1, fp.reduced_tx_set);
  int cands[16], nc = 0;
  if (plane == 0) {
    if (!fp.tx_search || set == TX_SET_DCTONLY || fp.lossless) cands[nc++] = DCT_DCT;
    else
      for (int t = 0; t < 16; t++)
        if (in_set(set, t, 1)) cands[nc++] = t;
  } else {
    int t = b.tx_type;
    if (Tx_Size_Sqr_Up[txSz] > TX_32X32 || !in_set(set, t, 1)) t = DCT_DCT;
    cands[nc++] = t;
  }
  int txIdx = 0, anyNz = 0;
  for (int y = 0; y < n4h; y += stepY)
    for (int x = 0; x < n4w; x += stepX) {
      const int sx = baseX + 4 * x, sy = baseY + 4 * y;
      if (sx >= ((fp.mi_cols * 4) >> sub) || sy >= ((fp.mi_rows * 4) >> sub)) continue;
      int t = DCT_DCT;
      long long c = 0;
      const int eob = code_tx_block(fp, spx, px, S, sx, sy, txSz, plane, cands, nc,
                                    coefs + b.coef_off[plane] + txIdx * Tx_Width[txSz] * Tx_Height[txSz], mats, &t, &c);
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
      __syncthreads();
    }
  if (tid == 0) b.eob[plane] = anyNz;
  __syncthreads();
}

/* recon_block (k_recon.h:293-394) for the inter block in L.blk. */
NOINL void recon_inter_block(const Mav1FrameParams &fp, const uint8_t *__restrict__ src, uint8_t *rec,
                             const uint8_t *__restrict__ ref, const uint8_t *__restrict__ gold,
                             int32_t *__restrict__ coefs, const int32_t *__restrict__ mats) {
  RLds &L = gL;
  Mav1BlockInfo &b = L.blk;
  const int tid = threadIdx.x;
  const int bs = b.bsize, comp = b.ref_frame1 > INTRA_FRAME;
  const uint8_t *r0 = b.ref_frame != LAST_FRAME ? gold : ref;
  if (tid == 0) {
    b.tx_depth = 0;
    b.interp_filter &= 0x30;
  }
  __syncthreads();
  if (fp.switchable_interp && !comp) {
    const int f = dual_filter_search(fp, r0, src);
    if (tid == 0) b.interp_filter = f;
    __syncthreads();
  }
  for (int plane = 0; plane < 3; plane++) {
    const int sub = plane > 0, S = fp.stride[plane];
    const int baseX = (b.mi_col >> sub) * 4, baseY = (b.mi_row >> sub) * 4;
    const int w = BLOCK_WIDTH(bs) >> sub, h = BLOCK_HEIGHT(bs) >> sub;
    if (comp) {
      CompLds &P = L.u.cp;
      predict_inter_plane(r0 + fp.offset[plane], S, fp.frame_w, fp.frame_h, baseX, baseY, w, h, b.mv_row, b.mv_col, sub,
                          b.interp_filter, nullptr, w, P.p0, 7, P.win, P.mid);
      /* the second prediction in bands of 16 rows, combined with the first */
      for (int yy = 0; yy < h; yy += 16) {
        const int hh = d_min(16, h - yy);
        predict_inter_plane(gold + fp.offset[plane], S, fp.frame_w, fp.frame_h, baseX, baseY + yy, w, hh, b.mv1_row,
                            b.mv1_col, sub, b.interp_filter, nullptr, w, P.p1, 7, P.win, P.mid);
        uint8_t *d = rec + fp.offset[plane] + (baseY + yy) * S + baseX;
        for (int k = tid; k < w * hh; k += RT) {
          const int i = k / w, j = k - i * w;
          d[i * S + j] = (uint8_t)d_clip1(d_round2(P.p0[(yy + i) * w + j] + P.p1[i * w + j], 5));
        }
        __syncthreads();
      }
    } else {
      predict_inter_plane(r0 + fp.offset[plane], S, fp.frame_w, fp.frame_h, baseX, baseY, w, h, b.mv_row, b.mv_col, sub,
                          b.interp_filter, rec + fp.offset[plane] + baseY * S + baseX, S, nullptr, 11, L.u.pr.win,
                          L.u.pr.mid[0]);
    }
    const int t = fp.lossless ? TX_4X4 : plane > 0 ? uv_tx_size(bs) : Max_Tx_Size_Rect[bs];
    code_inter_plane(fp, src, rec, coefs, mats, plane, t);
  }
}

/* The inter blocks of the frame as a work list: work[0] = count, work[1] =
 * the next entry to take, work[2 + i] = block index. */
__global__ void k_recon_list_reset(int *work) {
  if (threadIdx.x < 2) work[threadIdx.x] = 0;
}
DEVI void recon_list_body(const Mav1FrameParams &fp, const Mav1BlockInfo *__restrict__ blocks, const Mav1SbInfo *__restrict__ sbs, int *work, const int blk_x, const int blk_y, const int blk_z) {
  const int sb = blk_x, k = threadIdx.x;
  if (k >= sbs[sb].num_blocks) return;
  const int bi = sbs[sb].first_block + k;
  if (blocks[bi].is_inter) work[2 + atomicAdd(&work[0], 1)] = bi;
}
__global__ __launch_bounds__(64) void k_recon_list(const Mav1FrameParams fp, const Mav1BlockInfo *__restrict__ blocks,
                                                   const Mav1SbInfo *__restrict__ sbs, int *work) {
  recon_list_body(fp, blocks, sbs, work, blockIdx.x, blockIdx.y, blockIdx.z);
}

/* Inter phase: persistent workgroups take the inter blocks off the list
 * one at a time until it is empty. */
__global__ __launch_bounds__(RT) void k_recon_inter(const Mav1FrameParams fp, Mav1BlockInfo *__restrict__ blocks,
                                                    const uint8_t *__restrict__ src, uint8_t *rec,
                                                    const uint8_t *__restrict__ ref, const uint8_t *__restrict__ gold,
                                                    int32_t *__restrict__ coefs, const int32_t *__restrict__ mats,
                                                    int *work) {
  RLds &L = gL;
  const int tid = threadIdx.x;
  stage_tabs(tid, RT);
  stage_smats(fp, mats);
  const int count = work[0];
  for (;;) {
    if (tid == 0) L.ival[2] = atomicAdd(&work[1], 1);
    __syncthreads();
    const int idx = L.ival[2];
    __syncthreads();
    if (idx >= count) break;
    Mav1BlockInfo *g = blocks + work[2 + idx];
    if (tid < 27) ((int32_t *)&L.blk)[tid] = ((const int32_t *)g)[tid];
    __syncthreads();
    recon_inter_block(fp, src, rec, ref, gold, coefs, mats);
    if (tid < 27) ((int32_t *)g)[tid] = ((const int32_t *)&L.blk)[tid];
    __syncthreads();
  }
}

/* ---- intra phase: one dataflow launch ----
 * k_intra_sched lists the superblocks holding intra blocks in order of
 * T = column + 2 row, then row. Every superblock whose reconstruction another
 * one reads (left, above-left, above, above-right) has a smaller T, so the
 * list is a topological order of the dependencies. k_recon_intra's
 * workgroups take the list's superblocks one at a time (an atomic counter);
 * before coding one they wait for its neighbours in the same tile column
 * that hold intra blocks, and they publish each finished superblock with an
 * agent-scope release. A workgroup only waits for superblocks taken earlier
 * by running workgroups, so every wait ends; it is still bounded, and a
 * wait that runs out sets iwork[IW_ERR] instead of hanging.
 * iwork: [0] count, [1] next, [2] error, [4 ..] the list, then per
 * superblock "holds intra blocks", then per superblock "done". */
#define SCHED_T 512
#define SCHED_KEYS 20480 /* (sb_cols + 2 sb_rows) sb_rows, checked on the host */

DEVI void intra_sched_body(const Mav1FrameParams &fp, const Mav1BlockInfo *__restrict__ blocks, const Mav1SbInfo *__restrict__ sbs, int *__restrict__ iwork, const int blk_x, const int blk_y, const int blk_z) {
  __shared__ uint16_t dense[SCHED_KEYS];
  __shared__ int cnt[SCHED_T + 1];
  const int n = fp.sb_cols * fp.sb_rows, tid = threadIdx.x;
  const int K = (fp.sb_cols + 2 * fp.sb_rows) * fp.sb_rows;
  int *list = iwork + IW_HDR, *has = list + n, *done = has + n;
  for (int k = tid; k < K; k += SCHED_T) dense[k] = 0;
  __syncthreads();
  for (int sb = tid; sb < n; sb += SCHED_T) {
    int h = 0;
    for (int i = 0; i < sbs[sb].num_blocks; i++) h |= !blocks[sbs[sb].first_block + i].is_inter;
    has[sb] = h;
    done[sb] = 0;
    const int r = sb / fp.sb_cols, c = sb - r * fp.sb_cols;
    if (h) dense[(c + 2 * r) * fp.sb_rows + r] = (uint16_t)(sb + 1);
  }
  __syncthreads();
  /* compaction in key order: per thread a contiguous range of keys */
  const int C = (K + SCHED_T - 1) / SCHED_T, k0 = tid * C, k1 = d_min(K, k0 + C);
  int m = 0;
  for (int k = k0; k < k1; k++) m += dense[k] != 0;
  cnt[tid + 1] = m;
  __syncthreads();
  if (tid == 0) {
    cnt[0] = 0;
    for (int i = 1; i <= SCHED_T; i++) cnt[i] += cnt[i - 1];
    iwork[IW_COUNT] = cnt[SCHED_T];
    iwork[IW_NEXT] = 0;
    iwork[IW_ERR] = 0;
  }
  __syncthreads();
  int o = cnt[tid];
  for (int k = k0; k < k1; k++)
    if (dense[k]) list[o++] = dense[k] - 1;
}
__global__ __launch_bounds__(SCHED_T) void k_intra_sched(const Mav1FrameParams fp, const Mav1BlockInfo *__restrict__ blocks,
                                                        const Mav1SbInfo *__restrict__ sbs, int *__restrict__ iwork) {
  intra_sched_body(fp, blocks, sbs, iwork, blockIdx.x, blockIdx.y, blockIdx.z);
}

/* Edge filter types (src/encoder.c:319-346): smooth flags per mi, then per
 * block the above / left neighbours' flags into interp_filter bits 4 / 5. */
DEVI void edge_flags_body(const Mav1FrameParams &fp, const Mav1BlockInfo *__restrict__ blocks, const Mav1SbInfo *__restrict__ sbs, uint8_t *ys, uint8_t *uvs, const int blk_x, const int blk_y, const int blk_z) {
  const int sb = blk_x, lane = threadIdx.x;
  stage_tabs(lane, 64);
  __syncthreads();
  if (lane >= sbs[sb].num_blocks) return;
  const Mav1BlockInfo b = blocks[sbs[sb].first_block + lane];
  const int sy = !b.is_inter && (b.y_mode == SMOOTH_PRED || b.y_mode == SMOOTH_V_PRED || b.y_mode == SMOOTH_H_PRED);
  const int su = !b.is_inter && (b.uv_mode == SMOOTH_PRED || b.uv_mode == SMOOTH_V_PRED || b.uv_mode == SMOOTH_H_PRED);
  for (int r = b.mi_row; r < b.mi_row + Num_4x4_Blocks_High[b.bsize] && r < fp.mi_rows; r++)
    for (int c = b.mi_col; c < b.mi_col + Num_4x4_Blocks_Wide[b.bsize] && c < fp.mi_cols; c++) {
      ys[r * fp.mi_cols + c] = (uint8_t)sy;
      uvs[r * fp.mi_cols + c] = (uint8_t)su;
    }
}
__global__ __launch_bounds__(64) void k_edge_flags(const Mav1FrameParams fp, const Mav1BlockInfo *__restrict__ blocks,
                                                   const Mav1SbInfo *__restrict__ sbs, uint8_t *ys, uint8_t *uvs) {
  edge_flags_body(fp, blocks, sbs, ys, uvs, blockIdx.x, blockIdx.y, blockIdx.z);
}
DEVI void edge_types_body(const Mav1FrameParams &fp, Mav1BlockInfo *__restrict__ blocks, const Mav1SbInfo *__restrict__ sbs, const uint8_t *ys, const uint8_t *uvs, const int blk_x, const int blk_y, const int blk_z) {
  const int sb = blk_x, lane = threadIdx.x;
  if (lane >= sbs[sb].num_blocks) return;
  Mav1BlockInfo *b = &blocks[sbs[sb].first_block + lane];
  const int cols = fp.mi_cols, rows = fp.mi_rows, r = b->mi_row, c = b->mi_col;
  const int au = r > 0, al = c > tile_start(fp, c);
  const int fy = (au && ys[(r - 1) * cols + c]) || (al && ys[r * cols + c - 1]);
  const int fuv = (au && uvs[(r - 1) * cols + d_min(c + 1, cols - 1)]) || (al && uvs[d_min(r + 1, rows - 1) * cols + c - 1]);
  b->interp_filter = (b->interp_filter & 15) | fy << 4 | fuv << 5;
}
__global__ __launch_bounds__(64) void k_edge_types(const Mav1FrameParams fp, Mav1BlockInfo *__restrict__ blocks,
                                                   const Mav1SbInfo *__restrict__ sbs, const uint8_t *ys,
                                                   const uint8_t *uvs) {
  edge_types_body(fp, blocks, sbs, ys, uvs, blockIdx.x, blockIdx.y, blockIdx.z);
}

hipError_t launch_edge_types(hipStream_t st, const Mav1FrameParams &fp, Mav1BlockInfo *blocks, const Mav1SbInfo *sbs,
                             uint8_t *ys, uint8_t *uvs) {
  const int nsb = fp.sb_cols * fp.sb_rows;
  hipLaunchKernelGGL(k_edge_flags, dim3(nsb), dim3(64), 0, st, fp, blocks, sbs, ys, uvs);
  hipLaunchKernelGGL(k_edge_types, dim3(nsb), dim3(64), 0, st, fp, blocks, sbs, ys, uvs);
  return hipGetLastError();
}

hipError_t launch_recon_inter(hipStream_t st, const Mav1FrameParams &fp, Mav1BlockInfo *blocks, const Mav1SbInfo *sbs,
                              const uint8_t *src, uint8_t *rec, const uint8_t *ref, const uint8_t *gold,
                              int32_t *coefs, const int32_t *mats, int *work, int workgroups) {
  const int nsb = fp.sb_cols * fp.sb_rows;
  hipLaunchKernelGGL(k_recon_list_reset, dim3(1), dim3(64), 0, st, work);
  hipLaunchKernelGGL(k_recon_list, dim3(nsb), dim3(64), 0, st, fp, (const Mav1BlockInfo *)blocks, sbs, work);
  hipLaunchKernelGGL(k_recon_inter, dim3(workgroups), dim3(RT), 0, st, fp, blocks, src, rec, ref, gold, coefs, mats,
                     work);
  return hipGetLastError();
}


/* list, has, done and (batched form) the pending-dependency counts */
size_t intra_work_ints(const Mav1FrameParams &fp) { return IW_HDR + 4 * (size_t)fp.sb_cols * fp.sb_rows; }
/* Workgroups for the intra phase of one frame: twice the superblocks the
 * dependency order lets run at once (per tile column, one superblock in
 * every second column of a diagonal c + 2 r), at least 16, at most the CU
 * count. More only hold CUs while they wait, which the other streams'
 * kernels could use. */
int intra_workgroups(const Mav1FrameParams &fp, int num_cu) {
  const int tiles = (fp.sb_cols + fp.tile_w_sb - 1) / fp.tile_w_sb;
  const int per = ((fp.tile_w_sb < 2 * fp.sb_rows ? fp.tile_w_sb : 2 * fp.sb_rows) + 1) / 2;
  const int wg = 2 * tiles * per < 16 ? 16 : 2 * tiles * per;
  return wg < num_cu ? wg : num_cu;
}

int intra_sched_fits(const Mav1FrameParams &fp) {
  return (fp.sb_cols + 2 * fp.sb_rows) * fp.sb_rows <= SCHED_KEYS && fp.sb_cols * fp.sb_rows < 65535;
}

hipError_t launch_intra_sched(hipStream_t st, const Mav1FrameParams &fp, const Mav1BlockInfo *blocks,
                              const Mav1SbInfo *sbs, int *iwork) {
  hipLaunchKernelGGL(k_intra_sched, dim3(1), dim3(SCHED_T), 0, st, fp, blocks, sbs, iwork);
  return hipGetLastError();
}

/* Whether the frame's intra luma blocks search transform types or depths. */
__host__ DEVI bool intra_search(const Mav1FrameParams &fp) { return fp.tx_mode_select || fp.tx_search; }

hipError_t launch_recon_intra(hipStream_t st, const Mav1FrameParams &fp, Mav1BlockInfo *blocks, const Mav1SbInfo *sbs,
                              const uint8_t *src, uint8_t *rec, int32_t *coefs, const int32_t *mats, int *iwork,
                              int workgroups) {
  return (intra_search(fp) ? launch_recon_intra_search : launch_recon_intra_plain)(st, fp, blocks, sbs, src, rec, coefs,
                                                                                   mats, iwork, workgroups);
}

size_t intra_queue_ints(int qcap) { return 2 * (size_t)QH_INTS(qcap); }

int intra_searches(const BatchFrame *H, int n) {
  int search = 0;
  for (int f = 0; f < n; f++) search += intra_search(H[f].fp);
  return search;
}
hipError_t launch_recon_intra_b(hipStream_t st, const BatchFrame *T, int n, int *q, int qcap, int search,
                                int workgroups) {
  return search ? launch_recon_intra_search_b(st, T, n, q + QH_INTS(qcap), workgroups)
                : launch_recon_intra_plain_b(st, T, n, q, workgroups);
}

/* ---- batched launches (batch.h): the same kernels over several frames ---- */

__global__ __launch_bounds__(64) void k_edge_flags_b(const BatchFrame *__restrict__ T, const BatchGrid g) {
  const BatchIdx b = batch_idx(g);
  const BatchFrame &F = T[b.f];
  edge_flags_body(F.fp, gptr(F.blocks), gptr(F.sbs), gptr(F.ys), gptr(F.uvs), b.x, b.y, b.z);
}
__global__ __launch_bounds__(64) void k_edge_types_b(const BatchFrame *__restrict__ T, const BatchGrid g) {
  const BatchIdx b = batch_idx(g);
  const BatchFrame &F = T[b.f];
  edge_types_body(F.fp, gptr(F.blocks), gptr(F.sbs), gptr(F.ys), gptr(F.uvs), b.x, b.y, b.z);
}
__global__ void k_recon_list_reset_b(const BatchFrame *__restrict__ T) {
  if (threadIdx.x < 2) T[blockIdx.x].rwork[threadIdx.x] = 0;
}
__global__ __launch_bounds__(64) void k_recon_list_b(const BatchFrame *__restrict__ T, const BatchGrid g) {
  const BatchIdx b = batch_idx(g);
  const BatchFrame &F = T[b.f];
  recon_list_body(F.fp, gptr(F.blocks), gptr(F.sbs), gptr(F.rwork), b.x, b.y, b.z);
}

/* Inter phase over several frames: every workgroup takes the inter blocks
 * of frame 0 off its list until the list is empty, then frame 1's, and so
 * on; the frame-dependent LDS tables are staged when a workgroup takes its
 * first block of a frame. */
__global__ __launch_bounds__(RT) void k_recon_inter_b(const BatchFrame *__restrict__ T, int nfr) {
  RLds &L = gL;
  const int tid = threadIdx.x;
  stage_tabs(tid, RT);
  for (int f = 0; f < nfr; f++) {
    const BatchFrame &F = T[f];
    int *work = gptr(F.rwork);
    const int count = work[0];
    bool staged = false;
    for (;;) {
      if (tid == 0) L.ival[2] = atomicAdd(&work[1], 1);
      __syncthreads();
      const int idx = L.ival[2];
      __syncthreads();
      if (idx >= count) break;
      if (!staged) {
        stage_smats(F.fp, gptr(F.mats));
        __syncthreads();
        staged = true;
      }
      Mav1BlockInfo *gb = gptr(F.blocks) + work[2 + idx];
      if (tid < 27) ((int32_t *)&L.blk)[tid] = ((const int32_t *)gb)[tid];
      __syncthreads();
      recon_inter_block(F.fp, gptr(F.src), gptr(F.rec), gptr(F.ref), gptr(F.gold), gptr(F.coefs), gptr(F.mats));
      if (tid < 27) ((int32_t *)gb)[tid] = ((const int32_t *)&L.blk)[tid];
      __syncthreads();
    }
  }
}

__global__ __launch_bounds__(SCHED_T) void k_intra_sched_b(const BatchFrame *__restrict__ T) {
  const BatchFrame &F = T[blockIdx.x];
  intra_sched_body(F.fp, gptr(F.blocks), gptr(F.sbs), gptr(F.iwork), 0, 0, 0);
}

__global__ void k_intra_queue_reset_b(int *__restrict__ q, int cap) {
  const int n = QH_INTS(cap);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    q[i] = q[n + i] = i < QH_ITEMS ? 0 : -1;
}

/* Per frame (one workgroup each, after the scheduling pass): the pending
 * dependency count of every superblock holding intra blocks; those with none
 * are queued, in the queue of the frame's intra kernel. */
__global__ __launch_bounds__(256) void k_intra_ready_b(const BatchFrame *__restrict__ T, int *__restrict__ q, int qcap) {
  const int f = blockIdx.x;
  const BatchFrame &F = T[f];
  const Mav1FrameParams &fp = F.fp;
  if (intra_search(fp)) q += QH_INTS(qcap);
  const int n = fp.sb_cols * fp.sb_rows;
  const int *has = gptr(F.iwork) + IW_HDR + n;
  int *cnt = gptr(F.iwork) + IW_HDR + 3 * n;
  int mine = 0;
  for (int sb = threadIdx.x; sb < n; sb += blockDim.x) {
    if (!has[sb]) continue;
    int dep[4], k = 0;
    intra_deps(fp, sb, dep);
    for (int j = 0; j < 4; j++) k += dep[j] >= 0 && has[dep[j]];
    cnt[sb] = k;
    mine++;
  }
  __syncthreads(); /* every count stored before any superblock is queued */
  for (int sb = threadIdx.x; sb < n; sb += blockDim.x)
    if (has[sb] && cnt[sb] == 0) queue_push(q, f << 16 | sb);
  if (mine) atomicAdd(&q[QH_TOTAL], mine);
}

hipError_t launch_edge_types_b(hipStream_t st, const BatchFrame *T, const BatchFrame *H, int n) {
  BatchGrid g = batch_grid();
  for (int f = 0; f < n; f++) batch_grid_add(g, H[f].fp.sb_cols * H[f].fp.sb_rows, 1, 1);
  hipLaunchKernelGGL(k_edge_flags_b, dim3(g.start[n]), dim3(64), 0, st, T, g);
  hipLaunchKernelGGL(k_edge_types_b, dim3(g.start[n]), dim3(64), 0, st, T, g);
  return hipGetLastError();
}

hipError_t launch_recon_inter_b(hipStream_t st, const BatchFrame *T, const BatchFrame *H, int n, int workgroups) {
  BatchGrid g = batch_grid();
  for (int f = 0; f < n; f++) batch_grid_add(g, H[f].fp.sb_cols * H[f].fp.sb_rows, 1, 1);
  hipLaunchKernelGGL(k_recon_list_reset_b, dim3(n), dim3(64), 0, st, T);
  hipLaunchKernelGGL(k_recon_list_b, dim3(g.start[n]), dim3(64), 0, st, T, g);
  hipLaunchKernelGGL(k_recon_inter_b, dim3(workgroups), dim3(RT), 0, st, T, n);
  return hipGetLastError();
}

hipError_t launch_intra_sched_b(hipStream_t st, const BatchFrame *T, const BatchFrame *H, int n, int *q, int qcap) {
  int need = 0;
  for (int f = 0; f < n; f++) need += H[f].fp.sb_cols * H[f].fp.sb_rows;
  if (need > qcap || n > (1 << 14)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_intra_sched_b, dim3(n), dim3(SCHED_T), 0, st, T);
  hipLaunchKernelGGL(k_intra_queue_reset_b, dim3(std::min((QH_INTS(qcap) + 255) / 256, 1024)), dim3(256), 0, st, q, qcap);
  hipLaunchKernelGGL(k_intra_ready_b, dim3(n), dim3(256), 0, st, T, q, qcap);
  return hipGetLastError();
}
