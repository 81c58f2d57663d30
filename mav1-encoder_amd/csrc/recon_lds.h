/* Tables and working sets of the reconstruction kernels (recon.hip: inter
 * phase; recon_intra.h: intra phase). Each of the two defines its RLds (the
 * LDS of the workgroup that reconstructs a block or a superblock, gL) on top
 * of what is here, then includes recon_tx.h. */
#ifndef MAV1_RECON_LDS_H
#define MAV1_RECON_LDS_H

#include <algorithm>
#include <climits>

#include "dev_common.h"

/* The small AV1 tables that these kernels index with per-lane values live
 * in LDS: in constant memory each such lookup is a vector load through the
 * L2, and the stages chain several of them. Every workgroup copies them in
 * first (stage_tabs); the names below then refer to the copies. */
struct RTabs {
  int16_t m2a[13], dr[90], iek[15], n4w[22], n4h[22], maxRect[22], maxDepth[22], split[19], subs[88];
  int16_t txw[19], txh[19], txwl[19], txhl[19], sqr[19], sqrUp[19], rowShift[19], inIntra[48], inInter[64], m2t[14];
  uint8_t sw[124];
  unsigned long long candList[3]; /* per intra transform set its types in order, a nibble each, and their number */
  int candCnt[3];
};
__shared__ RTabs gT;
template <class T>
DEVI void tab_copy(int16_t *d, const T *s, int n, int tid, int nt) {
  for (int k = tid; k < n; k += nt) d[k] = (int16_t)s[k];
}
DEVI void stage_tabs(int tid, int nt) {
  tab_copy(gT.m2a, Mode_To_Angle, 13, tid, nt);
  tab_copy(gT.dr, Dr_Intra_Derivative, 90, tid, nt);
  tab_copy(gT.iek, Intra_Edge_Kernel, 15, tid, nt);
  tab_copy(gT.n4w, Num_4x4_Blocks_Wide, 22, tid, nt);
  tab_copy(gT.n4h, Num_4x4_Blocks_High, 22, tid, nt);
  tab_copy(gT.maxRect, Max_Tx_Size_Rect, 22, tid, nt);
  tab_copy(gT.maxDepth, Max_Tx_Depth, 22, tid, nt);
  tab_copy(gT.split, Split_Tx_Size, 19, tid, nt);
  tab_copy(gT.subs, Subsampled_Size, 88, tid, nt);
  tab_copy(gT.txw, Tx_Width, 19, tid, nt);
  tab_copy(gT.txh, Tx_Height, 19, tid, nt);
  tab_copy(gT.txwl, Tx_Width_Log2, 19, tid, nt);
  tab_copy(gT.txhl, Tx_Height_Log2, 19, tid, nt);
  tab_copy(gT.sqr, Tx_Size_Sqr, 19, tid, nt);
  tab_copy(gT.sqrUp, Tx_Size_Sqr_Up, 19, tid, nt);
  tab_copy(gT.rowShift, Transform_Row_Shift, 19, tid, nt);
  tab_copy(gT.inIntra, Tx_Type_In_Set_Intra, 48, tid, nt);
  tab_copy(gT.inInter, Tx_Type_In_Set_Inter, 64, tid, nt);
  tab_copy(gT.m2t, Mode_To_Txfm, 14, tid, nt);
  if (tid < 3) {
    unsigned long long l = 0;
    int n = 0;
    for (int t = 0; t < 16; t++)
      if (TX_IN_SET_INTRA(tid, t)) l |= (unsigned long long)t << (4 * n++);
    gT.candList[tid] = l;
    gT.candCnt[tid] = n;
  }
  const uint8_t *w[5] = {Sm_Weights_Tx_4x4, Sm_Weights_Tx_8x8, Sm_Weights_Tx_16x16, Sm_Weights_Tx_32x32,
                         Sm_Weights_Tx_64x64};
  for (int k = tid; k < 124; k += nt) {
    const int lg = k < 4 ? 0 : k < 12 ? 1 : k < 28 ? 2 : k < 60 ? 3 : 4, base = (4 << lg) - 4;
    gT.sw[k] = w[lg][k - base];
  }
}
#define Mode_To_Angle gT.m2a
#define Dr_Intra_Derivative gT.dr
#define Intra_Edge_Kernel gT.iek
#define Num_4x4_Blocks_Wide gT.n4w
#define Num_4x4_Blocks_High gT.n4h
#define Max_Tx_Size_Rect gT.maxRect
#define Max_Tx_Depth gT.maxDepth
#define Split_Tx_Size gT.split
#define Subsampled_Size gT.subs
#define Tx_Width gT.txw
#define Tx_Height gT.txh
#define Tx_Width_Log2 gT.txwl
#define Tx_Height_Log2 gT.txhl
#define Tx_Size_Sqr gT.sqr
#define Tx_Size_Sqr_Up gT.sqrUp
#define Transform_Row_Shift gT.rowShift
#define Tx_Type_In_Set_Intra gT.inIntra
#define Tx_Type_In_Set_Inter gT.inInter
#define Mode_To_Txfm gT.m2t
#define Sm_Weights_Tx_4x4 (gT.sw + 0)
#define Sm_Weights_Tx_8x8 (gT.sw + 4)
#define Sm_Weights_Tx_16x16 (gT.sw + 12)
#define Sm_Weights_Tx_32x32 (gT.sw + 28)
#define Sm_Weights_Tx_64x64 (gT.sw + 60)

#include "dev_pred.h"
#include "dev_tx.h"
#include "internal.h"

#define RT 512       /* threads of a reconstruction workgroup */
#define RW (RT / 64) /* its waves */
#define BDD 18
#define BDI(p, y, x) ((p) * BDD * BDD + ((y) + 1) * BDD + ((x) + 1))

#define SRS 17 /* row strides of a small (<= 16x16) block: residual, dequantised */
#define SQS 17
#define BRS 65 /* and of a large one */
#define BQS 33

/* One wave's working set for a transform block of at most 16x16. */
struct SmallTx {
  int32_t resid[16 * SRS]; /* residual, then the inverse transform's output */
  int32_t tmp[256];
  int32_t coef[256];
  int32_t q[256];
  int32_t dq[16 * SQS];
};
/* The workgroup's working set for a larger transform block. */
struct BigTx {
  int32_t resid[64 * BRS];
  int32_t tmp[64 * 32];
  int32_t coef[32 * 32];
  int32_t qtry[32 * 32];
  int32_t qbest[32 * 32];
  int32_t dq[32 * BQS];
};

/* The scans of the nine transform sizes up to 16x16, back to back. */
#define SCAN_SMALL 784

/* Work space of the intra phase (iwork): count, next, error word, then the
 * list, per superblock "holds intra blocks", "done" and (batched form) the
 * pending dependencies. */
#define IW_COUNT 0
#define IW_NEXT 1
#define IW_ERR 2
#define IW_HDR 4

/* What the transform stages use of a workgroup's LDS. */
struct RCommon {
  int32_t qbest[256];
  long long candCost[16];
  int candEob[16];
  long long red[RW];
  uint8_t tsrc[64 * 64], tpred[64 * 64]; /* the transform block's source and prediction */
  alignas(16) int32_t smats[TX_SMATS];
  int16_t scans[3 * SCAN_SMALL]; /* scans of the transforms up to 16x16: default, mrow, mcol */
  int16_t iscans[3 * SCAN_SMALL]; /* their inverses: the scan position of each coefficient */
  float qrcp[3][2];         /* per plane the quantiser reciprocals of dc_q / ac_q */
  int ival[4];
  Mav1BlockInfo blk;
};
#define NOINL __device__ __forceinline__

#endif
