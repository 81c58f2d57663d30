/* Learned partition / mode pruner: a small CNN trained and run on the GPU
 * with hand-written BF16 MFMA kernels (FP32 accumulation).
 *
 * No counterpart in the reference, whose analysis searches every partition
 * slot (src/kernels/k_analysis.h:656-679, the DP of :697-808) and inter
 * candidate (:256-311) exhaustively. The network predicts, per 64x64
 * superblock, a 4-way partition class and an 8-way inter-mode class from
 * the superblock's luma and its residual against the co-located reference
 * block, and the frame's quantiser.
 *
 * Network (activations NHWC, channels innermost):
 *   x0  64x64x2   luma / 255, residual / 255
 *   y1  32x32x32  ReLU(conv3x3 stride 2 pad 1 (x0) + b1)
 *   y2  16x16x64  ReLU(conv3x3 s2 p1 (y1) + b2)
 *   y3  8x8x64    ReLU(conv3x3 s2 p1 (y2) + b3)
 *   h   64        mean of y3 over the 8x8 positions + q * wq + bq
 *   partition logits h . Wp + bp (4), mode logits h . Wm + bm (8)
 *   loss: mean over the batch of the two softmax cross-entropies.
 * Conv operands (inputs, weights, the stored activations and the gradients
 * of the pre-activations) are BF16, rounded to nearest even; the products
 * accumulate in FP32 on the matrix cores (v_mfma_f32_16x16x32_bf16); the
 * pooling, heads, loss and the optimizer run in FP32.
 *
 * Each convolution is an implicit GEMM over 16x16x32 tiles:
 *   forward      out[co][pixel]  = sum_k W[co][k] im2col(in)[pixel][k]
 *   data grad    din[ci][pixel]  = sum_k Wt[ci][k] gather(dpre)[pixel][k]
 *   weight grad  dW[co][k]       = sum_pixel dpre[pixel][co] im2col(in)[pixel][k]
 * with k = tap * C + c (tap = 3 ky + kx). A workgroup carries a sample
 * through all layers in LDS (k_forward, k_backward); the weight gradients of
 * the workgroups are added in a fixed order, so every result is
 * deterministic. */
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include "../../include/mav1_hip.h"
#include "batch.h"

namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

/* parameter layout (FP32, flat): conv weights [co][tap][ci] */
constexpr int C0 = 2, C1 = 32, C2 = 64, C3 = 64, NP = 4, NM = 8, NF = 64;
constexpr int P_W1 = 0, P_B1 = P_W1 + C1 * 9 * C0, P_W2 = P_B1 + C1, P_B2 = P_W2 + C2 * 9 * C1, P_W3 = P_B2 + C2,
              P_B3 = P_W3 + C3 * 9 * C2, P_WQ = P_B3 + C3, P_BQ = P_WQ + NF, P_WP = P_BQ + NF, P_BP = P_WP + NF * NP,
              P_WM = P_BP + NP, P_BM = P_WM + NF * NM, P_N = P_BM + NM;
constexpr int K1 = 32;              /* 9 * C0 = 18 padded to a matrix instruction's 32 */
constexpr int K2 = 9 * C1, K3 = 9 * C2;
constexpr int MAX_SLICES = 256;     /* workgroups (and partial sums) of the weight gradients */

__device__ __forceinline__ uint16_t f2bf(float f) {
  /* round to nearest even on the upper 16 bits (finite inputs) */
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint32_t pack2(float a, float b) { return f2bf(a) | (uint32_t)f2bf(b) << 16; }

/* The value unchanged, opaque to the optimiser: what is derived from it is
 * not hoisted out of the loop over samples. */
__device__ __forceinline__ int local(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
/* An operand of the 16x16x32 matrix instruction: lane l holds row (column)
 * l & 15, k = 8 (l >> 4) .. + 7. The result's lane l holds column l & 15, rows
 * 4 (l >> 4) .. + 3. */
union Frag {
  bf8 v;
  s4 h[2];
  uint32_t w[4];
};
__device__ __forceinline__ f4 mfma(const Frag &a, const Frag &b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, c, 0, 0, 0);
}
__device__ __forceinline__ Frag frag(const uint16_t *p) { /* eight consecutive k (16-byte aligned) */
  Frag f;
  *(uint4 *)f.w = *(const uint4 *)p;
  return f;
}
/* Four pixels' 16 channels from LDS with rows and columns exchanged, per
 * group of 16 lanes: lane l names pixel (l & 15) >> 2 of the group's four and
 * channels 4 (l & 3) .. + 3, and gets channel l & 15 of the four pixels. */
__device__ __forceinline__ s4 tr_read(const uint16_t *p) {
  typedef __attribute__((address_space(3))) s4 lds_s4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p);
}
/* Operand with the channels in the rows (columns) and eight pixels per lane
 * in k: the lane's addresses for its group's first and last four. */
__device__ __forceinline__ Frag tr_frag(const uint16_t *p0, const uint16_t *p1) {
  Frag f;
  f.h[0] = tr_read(p0);
  f.h[1] = tr_read(p1);
  return f;
}

/* BF16 copies of the conv weights: W [co][Kp] with k = tap * Ci + ci, zero
 * where there is no parameter; Wt [ci][tap * Co + co] for the data gradients
 * of layers 2 and 3. */
__global__ void k_pack(const float *__restrict__ P, uint16_t *w1, uint16_t *w2, uint16_t *w3, uint16_t *wt2,
                       uint16_t *wt3) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < C1 * K1) {
    const int co = i / K1, k = i % K1;
    w1[i] = k < 9 * C0 ? f2bf(P[P_W1 + co * 9 * C0 + k]) : 0;
  }
  if (i < C2 * K2) {
    const int co = i / K2, k = i % K2, tap = k / C1, ci = k % C1;
    const uint16_t v = f2bf(P[P_W2 + (co * 9 + tap) * C1 + ci]);
    w2[i] = v;
    wt2[ci * (9 * C2) + tap * C2 + co] = v;
  }
  if (i < C3 * K3) {
    const int co = i / K3, k = i % K3, tap = k / C2, ci = k % C2;
    const uint16_t v = f2bf(P[P_W3 + (co * 9 + tap) * C2 + ci]);
    w3[i] = v;
    wt3[ci * (9 * C3) + tap * C3 + co] = v;
  }
}

/* x [b][64][64][2] float -> x0 the same in bf16, two pixels per thread */
__global__ void k_input(const float4 *__restrict__ x, uint2 *__restrict__ x0, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float4 v = x[i];
  x0[i] = make_uint2(pack2(v.x, v.y), pack2(v.z, v.w));
}

/* ---- a sample's activations in LDS ----
 * Pixel (y, x) at row y + 1, column x + 1: the row above and the column left
 * of the picture are the convolutions' zero padding (stride 2: nothing is
 * read below or right of it). Pixel strides of 80 and 144 bytes spread the
 * stride 2 gathers over the banks and keep 16-byte alignment. */
constexpr int PT = 512;              /* threads: 8 waves */
constexpr int X_W = 66;              /* x0 row in pixels (4 bytes each) */
constexpr int Y1_W = 33, Y1_S = 40;  /* row in pixels, pixel in halfwords */
constexpr int Y2_W = 17, Y2_S = 72;
struct FwdLds {
  alignas(16) uint32_t x0[65 * X_W];
  alignas(16) uint16_t y1[Y1_W * Y1_W * Y1_S];
  alignas(16) uint16_t y2[Y2_W * Y2_W * Y2_S];
  float part[2][C3];
};
/* A result tile's column (pixel) of four channels: bias, ReLU, BF16. */
__device__ __forceinline__ uint2 relu4(f4 v, f4 b) {
  float r[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const float t = v[j] + b[j];
    r[j] = t > 0.f ? t : 0.f;
  }
  return make_uint2(pack2(r[0], r[1]), pack2(r[2], r[3]));
}

/* The three convolutions and the pooling of samples blockIdx.x, + gridDim.x,
 * ..: one persistent workgroup per CU holds a sample's activations in LDS and
 * the weights in registers, so an inference reads the input and writes 64
 * means. hm [b][64]: the means; STORE: the activations too, for the backward
 * pass. A wave takes (conv1) every eighth tile of 16 pixels and all 32
 * channels, (conv2) 32 channels and four rows, (conv3) 16 channels and 32
 * pixels; the next sample's input is loaded during conv2.
 * Bound by the LDS reads of the pixel operand (each read by two matrix
 * instructions) and the barriers between the layers: 70 us for 2040 samples.
 * As three launches over global memory with 16 pixels and K = 16 a wave they
 * took 480 us. */
template <bool STORE>
__global__ __launch_bounds__(PT) void k_forward(const uint32_t *__restrict__ x0, const uint16_t *__restrict__ w1,
                                                const uint16_t *__restrict__ w2, const uint16_t *__restrict__ w3,
                                                const float *__restrict__ P, uint16_t *__restrict__ gy1,
                                                uint16_t *__restrict__ gy2, uint16_t *__restrict__ gy3,
                                                float *__restrict__ hm, int B) {
  __shared__ FwdLds S;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = lane & 15, kg0 = lane >> 4;
  int r = r0, kg = kg0;
  /* the wave's weights */
  const int ch = (wave & 1) * 32, rows = (wave >> 1) * 4, cot = (wave & 3) * 16, pt = (wave >> 2) * 2;
  Frag f1[2], f2[2][9], f3[18];
  f4 b1[2], b2[2], b3;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    f1[t] = frag(w1 + (t * 16 + r) * K1 + kg * 8);
#pragma unroll
    for (int k = 0; k < 9; k++) f2[t][k] = frag(w2 + (ch + t * 16 + r) * K2 + k * 32 + kg * 8);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      b1[t][j] = P[P_B1 + t * 16 + kg * 4 + j];
      b2[t][j] = P[P_B2 + ch + t * 16 + kg * 4 + j];
    }
  }
#pragma unroll
  for (int k = 0; k < 18; k++) f3[k] = frag(w3 + (cot + r) * K3 + k * 32 + kg * 8);
#pragma unroll
  for (int j = 0; j < 4; j++) b3[j] = P[P_B3 + cot + kg * 4 + j];
  /* conv1: the lane's four taps (4 kg ..) as offsets from the window's first pixel */
  int xo[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int tap = 4 * kg + i;
    xo[i] = tap < 9 ? (tap / 3) * X_W + tap % 3 : -1;
  }
  for (int i = tid; i < (int)(sizeof(FwdLds) / 4); i += PT) ((uint32_t *)&S)[i] = 0; /* the padding */
  uint4 nx[2] = {};
  auto fetch = [&](int b) {
#pragma unroll
    for (int i = 0; i < 2; i++) nx[i] = ((const uint4 *)(x0 + (size_t)b * 4096))[tid + i * PT];
  };
  fetch(blockIdx.x);
  for (int b = blockIdx.x; b < B; b += gridDim.x) {
    r = local(r0); /* the addresses are computed per sample, not kept in registers */
    kg = local(kg0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int q = (tid + i * PT) * 4;
      uint32_t *d = S.x0 + ((q >> 6) + 1) * X_W + (q & 63) + 1;
      d[0] = nx[i].x;
      d[1] = nx[i].y;
      d[2] = nx[i].z;
      d[3] = nx[i].w;
    }
    __syncthreads();
    for (int t = wave; t < 64; t += 8) {
      const int oy = t >> 1, ox = (t & 1) * 16 + r, base = 2 * oy * X_W + 2 * ox;
      Frag a;
#pragma unroll
      for (int i = 0; i < 4; i++) a.w[i] = S.x0[xo[i] >= 0 ? base + xo[i] : 0]; /* x0[0] is padding */
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const uint2 v = relu4(mfma(f1[c], a, f4{0.f, 0.f, 0.f, 0.f}), b1[c]);
        *(uint2 *)(S.y1 + ((oy + 1) * Y1_W + ox + 1) * Y1_S + c * 16 + kg * 4) = v;
        if (STORE) *(uint2 *)(gy1 + ((size_t)b * 1024 + oy * 32 + ox) * C1 + c * 16 + kg * 4) = v;
      }
    }
    __syncthreads();
    if (b + (int)gridDim.x < B) fetch(b + gridDim.x);
    {
      f4 acc[4][2];
#pragma unroll
      for (int t = 0; t < 4; t++) acc[t][0] = acc[t][1] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 9; k++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const Frag a = frag(S.y1 + ((2 * (rows + t) + k / 3) * Y1_W + 2 * r + k % 3) * Y1_S + kg * 8);
          acc[t][0] = mfma(f2[0][k], a, acc[t][0]);
          acc[t][1] = mfma(f2[1][k], a, acc[t][1]);
        }
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
          const uint2 v = relu4(acc[t][c], b2[c]);
          *(uint2 *)(S.y2 + ((rows + t + 1) * Y2_W + r + 1) * Y2_S + ch + c * 16 + kg * 4) = v;
          if (STORE) *(uint2 *)(gy2 + ((size_t)b * 256 + (rows + t) * 16 + r) * C2 + ch + c * 16 + kg * 4) = v;
        }
    }
    __syncthreads();
    {
      f4 acc[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int k = 0; k < 18; k++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
          const int oy = 2 * (pt + t) + (r >> 3), ox = r & 7, tap = k >> 1;
          const Frag a = frag(S.y2 + ((2 * oy + tap / 3) * Y2_W + 2 * ox + tap % 3) * Y2_S + (k & 1) * 32 + kg * 8);
          acc[t] = mfma(f3[k], a, acc[t]);
        }
      float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const uint2 v = relu4(acc[t], b3);
        if (STORE) *(uint2 *)(gy3 + ((size_t)b * 64 + (pt + t) * 16 + r) * C3 + cot + kg * 4) = v;
        s[0] += bf2f((uint16_t)v.x);
        s[1] += bf2f((uint16_t)(v.x >> 16));
        s[2] += bf2f((uint16_t)v.y);
        s[3] += bf2f((uint16_t)(v.y >> 16));
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) s[j] += __shfl_xor(s[j], o);
        if (r == j) S.part[wave >> 2][cot + kg * 4 + j] = s[j];
      }
    }
    __syncthreads();
    if (tid < C3) hm[(size_t)b * C3 + tid] = (S.part[0][tid] + S.part[1][tid]) / 64.f;
  }
}

/* ---- the convolutions' gradients ---- */
constexpr int D2_W = 18, D3_W = 9;
struct BwdLds {
  alignas(16) uint32_t x0[65 * X_W];
  alignas(16) uint16_t y1[Y1_W * Y1_W * Y1_S]; /* then d1 (in place) */
  alignas(16) uint16_t y2[D2_W * D2_W * Y2_S]; /* then d2 (in place), zeros below and right of it too */
  alignas(16) uint16_t d3[D3_W * D3_W * Y2_S]; /* from pixel (0, 0) on, zeros below and right of it */
};
static_assert(sizeof(BwdLds) <= 160 * 1024, "LDS");
/* The taps that reach an input coordinate of parity p: tap n's index k, and
 * the output coordinate e + add, for coordinate 2 e + p = 2 o - 1 + k. */
__device__ __forceinline__ constexpr int tap_k(int p, int n) { return p ? 2 * n : 1; }
__device__ __forceinline__ constexpr int tap_add(int p, int n) { return p && n == 0 ? 1 : 0; }
/* v where the activation y is positive, BF16 */
__device__ __forceinline__ uint2 mask4(f4 v, uint2 y) {
  const uint32_t a = pack2(v[0], v[1]), b = pack2(v[2], v[3]);
  const auto m = [](uint32_t w) { return (bf2f((uint16_t)w) > 0.f ? 0xFFFFu : 0u) | (bf2f((uint16_t)(w >> 16)) > 0.f ? 0xFFFF0000u : 0u); };
  return make_uint2(a & m(y.x), b & m(y.y));
}

/* Weight, bias and data gradients of samples blockIdx.x, + gridDim.x, ..: a
 * workgroup holds a sample's activations in LDS and, in turn, the
 * pre-activation gradients d3, d2 (over y2) and d1 (over y1); the weight
 * gradients stay in registers over the workgroup's samples and end as its
 * slice of part (parameter order, P_WQ floats). A weight gradient is a
 * product over the pixels, whose operands come from the pixel-major LDS
 * images by transposing reads; bias gradients are products with ones. A data
 * gradient gathers, per parity of the pixel's row and column, only the taps
 * that reach it (9 of 36 tap and parity pairs).
 * Bound by LDS reads and barriers of one workgroup per CU. As separate
 * launches over global memory the gradients of 256 samples took 1.93 ms
 * (weights 1.25, biases 0.43, data 0.26), here 40 us and 9 us for the sums of
 * the slices. */
__global__ __launch_bounds__(PT) void k_backward(const uint32_t *__restrict__ x0, const uint16_t *__restrict__ gy1,
                                                 const uint16_t *__restrict__ gy2, const uint16_t *__restrict__ gy3,
                                                 const float *__restrict__ dh, const uint16_t *__restrict__ wt2,
                                                 const uint16_t *__restrict__ wt3, float *__restrict__ part, int B) {
  __shared__ BwdLds S;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int r, kg, tp, tc; /* tr_read: pixel tp, channels tc .. */
  auto lanes = [&]() { /* addresses and weights are taken per phase, not kept in registers */
    const int l = local(lane);
    r = l & 15;
    kg = l >> 4;
    tp = (l & 15) >> 2;
    tc = (l & 3) * 4;
  };
  lanes();
  const f4 zero = {0.f, 0.f, 0.f, 0.f};
  f4 a3[5][4], a2[3][4], a1[2][2], ab3[4], ab2[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
#pragma unroll
    for (int i = 0; i < 5; i++) a3[i][c] = zero;
#pragma unroll
    for (int i = 0; i < 3; i++) a2[i][c] = zero;
    a1[c >> 1][c & 1] = ab3[c] = ab2[c] = zero;
  }
  Frag ones;
#pragma unroll
  for (int i = 0; i < 4; i++) ones.w[i] = 0x3F803F80u;
  for (int i = tid; i < (int)(sizeof(BwdLds) / 4); i += PT) ((uint32_t *)&S)[i] = 0;
  for (int b = blockIdx.x; b < B; b += gridDim.x) {
    __syncthreads();
    for (int q = tid; q < 1024; q += PT) {
      const uint4 v = ((const uint4 *)(x0 + (size_t)b * 4096))[q];
      uint32_t *d = S.x0 + ((q >> 4) + 1) * X_W + (q & 15) * 4 + 1;
      d[0] = v.x;
      d[1] = v.y;
      d[2] = v.z;
      d[3] = v.w;
    }
#pragma unroll 4
    for (int q = tid; q < 4096; q += PT) { /* 4 x 16 bytes per pixel */
      const int px = q >> 2;
      *(uint4 *)(S.y1 + ((px >> 5) + 1) * Y1_W * Y1_S + ((px & 31) + 1) * Y1_S + (q & 3) * 8) =
          ((const uint4 *)(gy1 + (size_t)b * 1024 * C1))[q];
    }
#pragma unroll
    for (int i = 0; i < 4; i++) { /* 8 x 16 bytes per pixel */
      const int q = tid + i * PT, px = q >> 3;
      *(uint4 *)(S.y2 + (((px >> 4) + 1) * D2_W + (px & 15) + 1) * Y2_S + (q & 7) * 8) =
          ((const uint4 *)(gy2 + (size_t)b * 256 * C2))[q];
    }
    {
      /* d3 = dh / 64 where y3 > 0 */
      const int px = tid >> 3, c = (tid & 7) * 8;
      const uint4 y = ((const uint4 *)(gy3 + (size_t)b * 64 * C3))[tid];
      const f4 g0 = *(const f4 *)(dh + (size_t)b * NF + c) / 64.f, g1 = *(const f4 *)(dh + (size_t)b * NF + c + 4) / 64.f;
      const uint2 lo = mask4(g0, make_uint2(y.x, y.y)), hi = mask4(g1, make_uint2(y.z, y.w));
      *(uint4 *)(S.d3 + ((px >> 3) * D3_W + (px & 7)) * Y2_S + c) = make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
    __syncthreads();
    lanes();
    /* layer 3 weights: column tiles (tap, 16 ci) wave + 8 i of 36, 2 x 32 pixels */
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      const int oy = ks * 4 + kg;
      Frag a[4];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const uint16_t *p = S.d3 + (oy * D3_W + tp) * Y2_S + c * 16 + tc;
        a[c] = tr_frag(p, p + 4 * Y2_S);
        if (wave == 7) ab3[c] = mfma(a[c], ones, ab3[c]);
      }
#pragma unroll
      for (int i = 0; i < 5; i++) {
        const int n = wave + 8 * i, tap = n >> 2;
        if (n < 36) {
          const uint16_t *p = S.y2 + ((2 * oy + tap / 3) * D2_W + 2 * tp + tap % 3) * Y2_S + (n & 3) * 16 + tc;
          const Frag v = tr_frag(p, p + 8 * Y2_S);
#pragma unroll
          for (int c = 0; c < 4; c++) a3[i][c] = mfma(a[c], v, a3[i][c]);
        }
      }
    }
    __syncthreads();
    lanes();
    /* d2 over y2: 16 ci per wave, two tiles of 16 pixels per parity class */
    {
      const int ct = (wave & 3) * 16, t0 = (wave >> 2) * 2;
#pragma unroll
      for (int cls = 0; cls < 4; cls++) {
        const int py = cls >> 1, qx = cls & 1;
        f4 acc[2] = {zero, zero};
#pragma unroll
        for (int ny = 0; ny < 1 + py; ny++)
#pragma unroll
          for (int nx = 0; nx < 1 + qx; nx++)
#pragma unroll
            for (int st = 0; st < 2; st++) {
              const int tap = tap_k(py, ny) * 3 + tap_k(qx, nx);
              const Frag w = frag(wt3 + (size_t)(ct + r) * (9 * C3) + tap * C3 + st * 32 + kg * 8);
#pragma unroll
              for (int t = 0; t < 2; t++) {
                const int oy = 2 * (t0 + t) + (r >> 3) + tap_add(py, ny), ox = (r & 7) + tap_add(qx, nx);
                acc[t] = mfma(w, frag(S.d3 + (oy * D3_W + ox) * Y2_S + st * 32 + kg * 8), acc[t]);
              }
            }
#pragma unroll
        for (int t = 0; t < 2; t++) {
          const int iy = 2 * (2 * (t0 + t) + (r >> 3)) + py, ix = 2 * (r & 7) + qx;
          uint2 *p = (uint2 *)(S.y2 + ((iy + 1) * D2_W + ix + 1) * Y2_S + ct + kg * 4);
          *p = mask4(acc[t], *p);
        }
      }
    }
    __syncthreads();
    lanes();
    /* layer 2 weights: column tiles wave + 8 i of 18, 8 x 32 pixels */
#pragma unroll 2
    for (int ks = 0; ks < 8; ks++) {
      const int oy = 2 * ks + (kg >> 1), ox = (kg & 1) * 8 + tp;
      Frag a[4];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const uint16_t *p = S.y2 + ((oy + 1) * D2_W + ox + 1) * Y2_S + c * 16 + tc;
        a[c] = tr_frag(p, p + 4 * Y2_S);
        if (wave == 7) ab2[c] = mfma(a[c], ones, ab2[c]);
      }
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const int n = wave + 8 * i, tap = n >> 1;
        if (n < 18) {
          const uint16_t *p = S.y1 + ((2 * oy + tap / 3) * Y1_W + 2 * ox + tap % 3) * Y1_S + (n & 1) * 16 + tc;
          const Frag v = tr_frag(p, p + 8 * Y1_S);
#pragma unroll
          for (int c = 0; c < 4; c++) a2[i][c] = mfma(a[c], v, a2[i][c]);
        }
      }
    }
    __syncthreads();
    lanes();
    /* d1 over y1: two rows of each parity class per wave, 32 ci */
#pragma unroll
    for (int cls = 0; cls < 4; cls++) {
      const int py = cls >> 1, qx = cls & 1;
      f4 acc[2][2] = {{zero, zero}, {zero, zero}};
#pragma unroll
      for (int ny = 0; ny < 1 + py; ny++)
#pragma unroll
        for (int nx = 0; nx < 1 + qx; nx++)
#pragma unroll
          for (int st = 0; st < 2; st++) {
            const int tap = tap_k(py, ny) * 3 + tap_k(qx, nx);
            const Frag w0 = frag(wt2 + (size_t)r * (9 * C2) + tap * C2 + st * 32 + kg * 8);
            const Frag w1 = frag(wt2 + (size_t)(16 + r) * (9 * C2) + tap * C2 + st * 32 + kg * 8);
#pragma unroll
            for (int t = 0; t < 2; t++) {
              const int oy = 2 * wave + t + tap_add(py, ny), ox = r + tap_add(qx, nx);
              const Frag v = frag(S.y2 + ((oy + 1) * D2_W + ox + 1) * Y2_S + st * 32 + kg * 8);
              acc[t][0] = mfma(w0, v, acc[t][0]);
              acc[t][1] = mfma(w1, v, acc[t][1]);
            }
          }
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
          const int iy = 2 * (2 * wave + t) + py, ix = 2 * r + qx;
          uint2 *p = (uint2 *)(S.y1 + ((iy + 1) * Y1_W + ix + 1) * Y1_S + c * 16 + kg * 4);
          *p = mask4(acc[t][c], *p);
        }
    }
    __syncthreads();
    lanes();
    /* layer 1 weights: columns 2 tap + ci, then a column of ones (the bias);
     * rows wave + 8 i, two column tiles */
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int oy = wave + 8 * i;
      Frag a[2], v[2];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const uint16_t *p = S.y1 + ((oy + 1) * Y1_W + kg * 8 + tp + 1) * Y1_S + c * 16 + tc;
        a[c] = tr_frag(p, p + 4 * Y1_S);
        const int col = c * 16 + r, tap = col < 18 ? col >> 1 : 0;
        const uint16_t *x = (const uint16_t *)S.x0 + (((2 * oy + tap / 3) * X_W + 2 * kg * 8 + tap % 3) * 2 + (col & 1));
#pragma unroll
        for (int q = 0; q < 8; q++) {
          const short e = (short)x[4 * q];
          v[c].h[q >> 2][q & 3] = col < 18 ? e : (short)(col == 18 ? 0x3F80 : 0);
        }
      }
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int n = 0; n < 2; n++) a1[c][n] = mfma(a[c], v[n], a1[c][n]);
    }
  }
  lanes();
  /* the workgroup's slice */
  float *o = part + (size_t)blockIdx.x * P_WQ;
#pragma unroll
  for (int c = 0; c < 4; c++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int co = c * 16 + kg * 4 + j;
#pragma unroll
      for (int i = 0; i < 5; i++) {
        const int n = wave + 8 * i;
        if (n < 36) o[P_W3 + (co * 9 + (n >> 2)) * C2 + (n & 3) * 16 + r] = a3[i][c][j];
      }
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const int n = wave + 8 * i;
        if (n < 18) o[P_W2 + (co * 9 + (n >> 1)) * C1 + (n & 1) * 16 + r] = a2[i][c][j];
      }
      if (wave == 7 && r == 0) {
        o[P_B3 + co] = ab3[c][j];
        o[P_B2 + co] = ab2[c][j];
      }
    }
  /* layer 1: the waves' sums in order */
  __syncthreads();
  float *red = (float *)S.y1; /* [wave][co][32] */
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int n = 0; n < 2; n++)
#pragma unroll
      for (int j = 0; j < 4; j++) red[(wave * 32 + c * 16 + kg * 4 + j) * 32 + n * 16 + r] = a1[c][n][j];
  __syncthreads();
  for (int i = tid; i < 32 * 32; i += PT) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < 8; w++) s += red[w * 1024 + i];
    const int co = i >> 5, col = i & 31;
    if (col < 18) o[P_W1 + co * 18 + col] = s;
    if (col == 18) o[P_B1 + co] = s;
  }
}

/* The slices added into the FP32 gradient: 64 parameters per block, a wave
 * per quarter of the slices, in a fixed order. */
__global__ __launch_bounds__(256) void k_slice_sum(const float *__restrict__ part, float *__restrict__ G, int n) {
  __shared__ float red[4][64];
  const int i = blockIdx.x * 64 + (threadIdx.x & 63), w = threadIdx.x >> 6;
  float s = 0.f;
  if (i < P_WQ) {
    const int z1 = n * (w + 1) / 4;
#pragma unroll 8
    for (int z = n * w / 4; z < z1; z++) s += part[(size_t)z * P_WQ + i];
  }
  red[w][threadIdx.x & 63] = s;
  __syncthreads();
  if (w == 0 && i < P_WQ) G[i] = (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
}

__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

/* Heads, one wave per sample (a lane per feature): features, logits, the
 * sample's loss (softmax cross-entropy of both heads, labels < 0 count
 * nothing). */
__global__ __launch_bounds__(256) void k_head_fwd(const float *__restrict__ hm, const float *__restrict__ q,
                                                  const float *__restrict__ P, const int *__restrict__ labels,
                                                  float *__restrict__ h, float *__restrict__ logits,
                                                  float *__restrict__ loss, int B) {
  const int b = blockIdx.x * 4 + (threadIdx.x >> 6), c = threadIdx.x & 63;
  if (b >= B) return;
  const float hv = hm[(size_t)b * NF + c] + q[b] * P[P_WQ + c] + P[P_BQ + c];
  h[(size_t)b * NF + c] = hv;
  float lg[NP + NM];
#pragma unroll
  for (int j = 0; j < NP; j++) lg[j] = wave_sum_f(hv * P[P_WP + c * NP + j]) + P[P_BP + j];
#pragma unroll
  for (int j = 0; j < NM; j++) lg[NP + j] = wave_sum_f(hv * P[P_WM + c * NM + j]) + P[P_BM + j];
  float z = 0.f;
#pragma unroll
  for (int j = 0; j < NP + NM; j++) z = c == j ? lg[j] : z;
  if (c < NP + NM) logits[(size_t)b * (NP + NM) + c] = z;
  float L = 0.f;
#pragma unroll
  for (int head = 0; head < 2; head++) {
    const int base = head ? NP : 0, n = head ? NM : NP, y = labels[2 * b + head];
    float mx = lg[base], ly = lg[base];
#pragma unroll
    for (int j = 1; j < n; j++) {
      mx = fmaxf(mx, lg[base + j]);
      ly = y == j ? lg[base + j] : ly;
    }
    float se = 0.f;
#pragma unroll
    for (int j = 0; j < n; j++) se += expf(lg[base + j] - mx);
    if (y >= 0) L += logf(se) + mx - ly;
  }
  if (c == 0) loss[b] = L;
}

__global__ __launch_bounds__(256) void k_loss_sum(const float *__restrict__ per, float *__restrict__ out, int B) {
  __shared__ float red[4];
  float s = 0.f;
  for (int b = threadIdx.x; b < B; b += 256) s += per[b];
  s = wave_sum_f(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[0] = ((red[0] + red[1]) + (red[2] + red[3])) / B;
}

/* Head backward per sample (a wave): d logits = (softmax - onehot) / B, and
 * the features' gradient dh. */
__global__ __launch_bounds__(256) void k_head_bwd(const float *__restrict__ logits, const int *__restrict__ labels,
                                                  const float *__restrict__ P, float *__restrict__ dlog,
                                                  float *__restrict__ dh, int B) {
  const int b = blockIdx.x * 4 + (threadIdx.x >> 6), c = threadIdx.x & 63;
  if (b >= B) return;
  const float *lg = logits + (size_t)b * (NP + NM);
  float g = 0.f, mine = 0.f;
#pragma unroll
  for (int head = 0; head < 2; head++) {
    const int base = head ? NP : 0, n = head ? NM : NP, y = labels[2 * b + head];
    float mx = lg[base];
#pragma unroll
    for (int j = 1; j < n; j++) mx = fmaxf(mx, lg[base + j]);
    float se = 0.f;
#pragma unroll
    for (int j = 0; j < n; j++) se += expf(lg[base + j] - mx);
#pragma unroll
    for (int j = 0; j < n; j++) {
      const float d = y < 0 ? 0.f : (expf(lg[base + j] - mx) / se - (j == y ? 1.f : 0.f)) / B;
      g += d * (head ? P[P_WM + c * NM + j] : P[P_WP + c * NP + j]);
      mine = c == base + j ? d : mine;
    }
  }
  if (c < NP + NM) dlog[(size_t)b * (NP + NM) + c] = mine;
  dh[(size_t)b * NF + c] = g;
}

/* Head parameter gradients, one wave per parameter, summed over the batch. */
__global__ __launch_bounds__(256) void k_head_grads(const float *__restrict__ h, const float *__restrict__ q,
                                                    const float *__restrict__ dlog, const float *__restrict__ dh,
                                                    float *__restrict__ G, int B) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  /* the parameter's two factors per sample: features (column f, or 1), then
   * d logits or dh (column j); q with dh */
  int f = -1, j = 0, kind = 0, out = 0; /* kind: 0 d logits, 1 dh, 2 dh * q */
  int t = i;
  if (t < NF * NP) {
    f = t / NP;
    j = t % NP;
    out = P_WP + t;
  } else if ((t -= NF * NP) < NP) {
    j = t;
    out = P_BP + t;
  } else if ((t -= NP) < NF * NM) {
    f = t / NM;
    j = NP + t % NM;
    out = P_WM + t;
  } else if ((t -= NF * NM) < NM) {
    j = NP + t;
    out = P_BM + t;
  } else if ((t -= NM) < NF) {
    j = t;
    kind = 2;
    out = P_WQ + t;
  } else if ((t -= NF) < NF) {
    j = t;
    kind = 1;
    out = P_BQ + t;
  } else {
    return;
  }
  float s = 0.f;
  for (int b = lane; b < B; b += 64) {
    const float d = kind ? dh[(size_t)b * NF + j] : dlog[(size_t)b * (NP + NM) + j];
    s += d * (kind == 2 ? q[b] : f >= 0 ? h[(size_t)b * NF + f] : 1.f);
  }
  s = wave_sum_f(s);
  if (lane == 0) G[out] = s;
}

__global__ void k_adam(float *__restrict__ P, const float *__restrict__ G, float *__restrict__ m1, float *__restrict__ m2,
                       float lr, float b1, float b2, float eps, float c1, float c2, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float g = G[i];
  const float a = b1 * m1[i] + (1.f - b1) * g, v = b2 * m2[i] + (1.f - b2) * g * g;
  m1[i] = a;
  m2[i] = v;
  P[i] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
}

/* A sample per superblock of the round's frames, straight from HBM: luma /
 * 255 and (inter frames) luma minus the LAST reference's co-located luma /
 * 255, as the training samples are built; q = base_q_idx / 255. */
__global__ __launch_bounds__(256) void k_frame_input(const BatchFrame *__restrict__ T, const BatchGrid g,
                                                     uint32_t *__restrict__ x0, float *__restrict__ q) {
  const BatchIdx b = batch_idx(g);
  const BatchFrame &F = T[b.f];
  const Mav1FrameParams &fp = F.fp;
  const int sr = b.x / fp.sb_cols, sc = b.x - sr * fp.sb_cols, S = fp.stride[0];
  const uint8_t *Y = F.src + fp.offset[0];
  const uint8_t *R = fp.frame_is_intra ? nullptr : F.ref + fp.offset[0];
  for (int pix = threadIdx.x; pix < 4096; pix += 256) {
    const int o = (sr * 64 + (pix >> 6)) * S + sc * 64 + (pix & 63);
    const int l = Y[o];
    x0[(size_t)blockIdx.x * 4096 + pix] = pack2((float)l / 255.f, R ? (float)(l - (int)R[o]) / 255.f : 0.f);
  }
  if (threadIdx.x == 0) q[blockIdx.x] = (float)fp.base_q_idx / 255.f;
}

__global__ void k_prune_levels(const BatchFrame *__restrict__ T, const BatchGrid g, const float *__restrict__ logits,
                               float tau) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= g.start[g.n]) return;
  const BatchIdx b = batch_idx(g, s);
  const BatchFrame &F = T[b.f];
  const Mav1FrameParams &fp = F.fp;
  const int sr = b.x / fp.sb_cols, sc = b.x - sr * fp.sb_cols;
  int lvl = 3;
  if ((sr + 1) * 16 <= fp.mi_rows && (sc + 1) * 16 <= fp.mi_cols) {
    const float *lg = logits + (size_t)s * (NP + NM);
    float mx = lg[0];
    for (int j = 1; j < NP; j++) mx = fmaxf(mx, lg[j]);
    float e[NP], se = 0.f;
    for (int j = 0; j < NP; j++) se += (e[j] = expf(lg[j] - mx));
    float cdf = 0.f;
    for (int l = 0; l < 3; l++) {
      cdf += e[l] / se;
      if (cdf >= 1.f - tau) {
        lvl = l;
        break;
      }
    }
  }
  F.prune[b.x] = (int8_t)lvl;
}

}  // namespace

struct mav1hip_pruner {
  int max_batch = 0, batch = 0;
  char err[256] = {0};
  hipStream_t st = nullptr;
  float *P = nullptr, *G = nullptr, *m1 = nullptr, *m2 = nullptr;
  uint16_t *w1 = nullptr, *w2 = nullptr, *w3 = nullptr, *wt2 = nullptr, *wt3 = nullptr;
  float *x = nullptr, *q = nullptr;
  int *labels = nullptr;
  uint32_t *x0 = nullptr; /* two bf16 per pixel */
  uint16_t *y1 = nullptr, *y2 = nullptr, *y3 = nullptr;
  float *hm = nullptr, *h = nullptr, *logits = nullptr, *dlog = nullptr, *dh = nullptr, *lossb = nullptr;
  float *loss = nullptr, *part = nullptr;
  int slices = 1; /* workgroups of k_forward and k_backward: one per CU */
  int packed = 0, forwarded = 0, labelled = 0;
};

namespace {

int pfail(mav1hip_pruner *p, int code, const char *fmt, ...) {
  if (p) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(p->err, sizeof p->err, fmt, ap);
    va_end(ap);
  }
  return code;
}

#define PCHK(p, call)                                                                                      \
  do {                                                                                                     \
    hipError_t e_ = (call);                                                                                \
    if (e_ != hipSuccess) return pfail(p, MAV1HIP_EDEVICE, "%s: %s (%s:%d)", #call, hipGetErrorString(e_), \
                                       __FILE__, __LINE__);                                                \
  } while (0)

template <class T>
int palloc(mav1hip_pruner *p, T **ptr, size_t n) {
  PCHK(p, hipMalloc((void **)ptr, n * sizeof(T)));
  PCHK(p, hipMemset(*ptr, 0, n * sizeof(T)));
  return MAV1HIP_OK;
}

int pack(mav1hip_pruner *p) {
  if (p->packed) return MAV1HIP_OK;
  const int n = C3 * K3;
  hipLaunchKernelGGL(k_pack, dim3((n + 255) / 256), dim3(256), 0, p->st, p->P, p->w1, p->w2, p->w3, p->wt2, p->wt3);
  PCHK(p, hipGetLastError());
  p->packed = 1;
  return MAV1HIP_OK;
}

/* Convolutions, pooling and heads of the batch; store: keep the activations
 * for the backward pass. */
int forward(mav1hip_pruner *p, bool store) {
  const dim3 grid(p->batch < p->slices ? p->batch : p->slices);
  if (store)
    hipLaunchKernelGGL(k_forward<true>, grid, dim3(PT), 0, p->st, p->x0, p->w1, p->w2, p->w3, p->P, p->y1, p->y2, p->y3,
                       p->hm, p->batch);
  else
    hipLaunchKernelGGL(k_forward<false>, grid, dim3(PT), 0, p->st, p->x0, p->w1, p->w2, p->w3, p->P, p->y1, p->y2,
                       p->y3, p->hm, p->batch);
  hipLaunchKernelGGL(k_head_fwd, dim3((p->batch + 3) / 4), dim3(256), 0, p->st, p->hm, p->q, p->P, p->labels, p->h,
                     p->logits, p->lossb, p->batch);
  PCHK(p, hipGetLastError());
  return MAV1HIP_OK;
}

void destroy_pruner(mav1hip_pruner *p) {
  if (!p) return;
  if (p->st) (void)hipStreamSynchronize(p->st);
  void *bufs[] = {p->P,  p->G,  p->m1, p->m2, p->w1, p->w2,     p->w3,   p->wt2, p->wt3,   p->x,    p->q,   p->labels,
                  p->x0, p->y1, p->y2, p->y3, p->h,  p->logits, p->dlog, p->dh,  p->lossb, p->loss, p->part, p->hm};
  for (void *b : bufs) (void)hipFree(b);
  if (p->st) (void)hipStreamDestroy(p->st);
  delete p;
}

}  // namespace

int pruner_infer_frames(mav1hip_pruner *p, hipStream_t st, const BatchFrame *T, const BatchFrame *H, int n, float tau) {
  if (!p || n < 1) return MAV1HIP_EINVAL;
  BatchGrid g = batch_grid();
  for (int f = 0; f < n; f++) batch_grid_add(g, H[f].fp.sb_cols * H[f].fp.sb_rows, 1, 1);
  const int total = g.start[n];
  if (total > p->max_batch) return pfail(p, MAV1HIP_EINVAL, "pruner: %d superblocks, room for %d", total, p->max_batch);
  hipStream_t own = p->st;
  p->st = st;
  p->batch = total;
  p->forwarded = 0; /* the loaded batch's inputs and features are overwritten: no backward pass on them */
  int rc = pack(p);
  if (!rc) {
    hipLaunchKernelGGL(k_frame_input, dim3(total), dim3(256), 0, st, T, g, p->x0, p->q);
    rc = hipGetLastError() == hipSuccess ? MAV1HIP_OK : pfail(p, MAV1HIP_EDEVICE, "pruner input launch failed");
  }
  if (!rc) rc = forward(p, false);
  if (!rc) {
    hipLaunchKernelGGL(k_prune_levels, dim3((total + 255) / 256), dim3(256), 0, st, T, g, p->logits, tau);
    rc = hipGetLastError() == hipSuccess ? MAV1HIP_OK : pfail(p, MAV1HIP_EDEVICE, "pruner launch failed");
  }
  p->st = own;
  return rc;
}

extern "C" {

int32_t mav1hip_pruner_num_params(void) { return P_N; }

mav1hip_pruner *mav1hip_pruner_create(int32_t max_batch, char *err, size_t errlen) {
  if (max_batch < 1 || max_batch > 4096) {
    if (err && errlen) snprintf(err, errlen, "max_batch must be 1 .. 4096");
    return nullptr;
  }
  mav1hip_pruner *p = new mav1hip_pruner();
  p->max_batch = max_batch;
  const size_t B = (size_t)max_batch;
  int rc = hipStreamCreate(&p->st) == hipSuccess ? MAV1HIP_OK : pfail(p, MAV1HIP_EDEVICE, "hipStreamCreate failed");
  int dev = 0, cus = 0;
  if (!rc && (hipGetDevice(&dev) != hipSuccess ||
              hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1))
    rc = pfail(p, MAV1HIP_EDEVICE, "device attributes");
  p->slices = cus < 1 ? 1 : cus < MAX_SLICES ? cus : MAX_SLICES;
  if (!rc) rc = palloc(p, &p->P, P_N);
  if (!rc) rc = palloc(p, &p->G, P_N);
  if (!rc) rc = palloc(p, &p->m1, P_N);
  if (!rc) rc = palloc(p, &p->m2, P_N);
  if (!rc) rc = palloc(p, &p->w1, (size_t)C1 * K1);
  if (!rc) rc = palloc(p, &p->w2, (size_t)C2 * K2);
  if (!rc) rc = palloc(p, &p->w3, (size_t)C3 * K3);
  if (!rc) rc = palloc(p, &p->wt2, (size_t)C1 * 9 * C2);
  if (!rc) rc = palloc(p, &p->wt3, (size_t)C2 * 9 * C3);
  if (!rc) rc = palloc(p, &p->x, B * 64 * 64 * C0);
  if (!rc) rc = palloc(p, &p->q, B);
  if (!rc) rc = palloc(p, &p->labels, 2 * B);
  if (!rc) rc = palloc(p, &p->x0, B * 64 * 64);
  if (!rc) rc = palloc(p, &p->y1, B * 32 * 32 * C1);
  if (!rc) rc = palloc(p, &p->y2, B * 16 * 16 * C2);
  if (!rc) rc = palloc(p, &p->y3, B * 8 * 8 * C3);
  if (!rc) rc = palloc(p, &p->hm, B * NF);
  if (!rc) rc = palloc(p, &p->h, B * NF);
  if (!rc) rc = palloc(p, &p->logits, B * (NP + NM));
  if (!rc) rc = palloc(p, &p->dlog, B * (NP + NM));
  if (!rc) rc = palloc(p, &p->dh, B * NF);
  if (!rc) rc = palloc(p, &p->lossb, B);
  if (!rc) rc = palloc(p, &p->loss, 1);
  if (!rc) rc = palloc(p, &p->part, (size_t)(max_batch < p->slices ? max_batch : p->slices) * P_WQ);
  if (rc) {
    if (err && errlen) snprintf(err, errlen, "%s", p->err);
    destroy_pruner(p);
    return nullptr;
  }
  return p;
}

void mav1hip_pruner_destroy(mav1hip_pruner *p) { destroy_pruner(p); }

const char *mav1hip_pruner_error(const mav1hip_pruner *p) { return p ? p->err : "no pruner"; }

int mav1hip_pruner_set_params(mav1hip_pruner *p, const float *params) {
  if (!p || !params) return MAV1HIP_EINVAL;
  PCHK(p, hipMemcpyAsync(p->P, params, sizeof(float) * P_N, hipMemcpyHostToDevice, p->st));
  PCHK(p, hipMemsetAsync(p->m1, 0, sizeof(float) * P_N, p->st));
  PCHK(p, hipMemsetAsync(p->m2, 0, sizeof(float) * P_N, p->st));
  PCHK(p, hipStreamSynchronize(p->st));
  p->packed = 0;
  return MAV1HIP_OK;
}

int mav1hip_pruner_get_params(mav1hip_pruner *p, float *params) {
  if (!p || !params) return MAV1HIP_EINVAL;
  PCHK(p, hipMemcpyAsync(params, p->P, sizeof(float) * P_N, hipMemcpyDeviceToHost, p->st));
  PCHK(p, hipStreamSynchronize(p->st));
  return MAV1HIP_OK;
}

int mav1hip_pruner_load(mav1hip_pruner *p, const float *x, const float *q, const int32_t *labels, int32_t batch) {
  if (!p || !x || !q || batch < 1 || batch > p->max_batch) return pfail(p, MAV1HIP_EINVAL, "load: bad batch");
  if (labels)
    for (int b = 0; b < batch; b++)
      if (labels[2 * b] < -1 || labels[2 * b] >= NP || labels[2 * b + 1] < -1 || labels[2 * b + 1] >= NM)
        return pfail(p, MAV1HIP_EINVAL, "load: sample %d has labels %d, %d (partition 0..3, mode 0..7, -1 none)", b,
                     labels[2 * b], labels[2 * b + 1]);
  p->batch = batch;
  PCHK(p, hipMemcpyAsync(p->x, x, sizeof(float) * (size_t)batch * 64 * 64 * C0, hipMemcpyHostToDevice, p->st));
  PCHK(p, hipMemcpyAsync(p->q, q, sizeof(float) * (size_t)batch, hipMemcpyHostToDevice, p->st));
  if (labels)
    PCHK(p, hipMemcpyAsync(p->labels, labels, sizeof(int32_t) * 2 * (size_t)batch, hipMemcpyHostToDevice, p->st));
  else
    PCHK(p, hipMemsetAsync(p->labels, 0xFF, sizeof(int32_t) * 2 * (size_t)batch, p->st));
  const int n = batch * 64 * 64 / 2;
  hipLaunchKernelGGL(k_input, dim3((n + 255) / 256), dim3(256), 0, p->st, (const float4 *)p->x, (uint2 *)p->x0, n);
  PCHK(p, hipGetLastError());
  p->forwarded = 0;
  p->labelled = labels != nullptr;
  return MAV1HIP_OK;
}

int mav1hip_pruner_forward(mav1hip_pruner *p, float *logits, float *loss) {
  if (!p || p->batch < 1) return pfail(p, MAV1HIP_EINVAL, "forward: no batch loaded");
  int rc;
  if ((rc = pack(p))) return rc;
  /* the activations are for the backward pass, whose gradients are zero without labels */
  if ((rc = forward(p, p->labelled))) return rc;
  hipLaunchKernelGGL(k_loss_sum, dim3(1), dim3(256), 0, p->st, p->lossb, p->loss, p->batch);
  PCHK(p, hipGetLastError());
  if (logits)
    PCHK(p, hipMemcpyAsync(logits, p->logits, sizeof(float) * (NP + NM) * (size_t)p->batch, hipMemcpyDeviceToHost,
                           p->st));
  if (loss) PCHK(p, hipMemcpyAsync(loss, p->loss, sizeof(float), hipMemcpyDeviceToHost, p->st));
  if (logits || loss) PCHK(p, hipStreamSynchronize(p->st));
  p->forwarded = 1;
  return MAV1HIP_OK;
}

int mav1hip_pruner_backward(mav1hip_pruner *p, float *grads) {
  if (!p || !p->forwarded) return pfail(p, MAV1HIP_EINVAL, "backward: run forward first");
  hipLaunchKernelGGL(k_head_bwd, dim3((p->batch + 3) / 4), dim3(256), 0, p->st, p->logits, p->labels, p->P, p->dlog,
                     p->dh, p->batch);
  hipLaunchKernelGGL(k_head_grads, dim3((NF * NP + NP + NF * NM + NM + 2 * NF + 3) / 4), dim3(256), 0, p->st, p->h,
                     p->q, p->dlog, p->dh, p->G, p->batch);
  /* without labels the forward pass kept no activations: no slices, so the sums are zeros */
  const int n = !p->labelled ? 0 : p->batch < p->slices ? p->batch : p->slices;
  if (n)
    hipLaunchKernelGGL(k_backward, dim3(n), dim3(PT), 0, p->st, p->x0, p->y1, p->y2, p->y3, p->dh, p->wt2, p->wt3,
                       p->part, p->batch);
  hipLaunchKernelGGL(k_slice_sum, dim3((P_WQ + 63) / 64), dim3(256), 0, p->st, p->part, p->G, n);
  PCHK(p, hipGetLastError());
  if (grads) {
    PCHK(p, hipMemcpyAsync(grads, p->G, sizeof(float) * P_N, hipMemcpyDeviceToHost, p->st));
    PCHK(p, hipStreamSynchronize(p->st));
  }
  return MAV1HIP_OK;
}

int mav1hip_pruner_adam(mav1hip_pruner *p, float lr, float beta1, float beta2, float eps, int32_t step) {
  if (!p || step < 1) return MAV1HIP_EINVAL;
  const float c1 = 1.f - powf(beta1, (float)step), c2 = 1.f - powf(beta2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3((P_N + 255) / 256), dim3(256), 0, p->st, p->P, p->G, p->m1, p->m2, lr, beta1, beta2,
                     eps, c1, c2, P_N);
  PCHK(p, hipGetLastError());
  p->packed = 0;
  return MAV1HIP_OK;
}

int mav1hip_pruner_sync(mav1hip_pruner *p) {
  if (!p) return MAV1HIP_EINVAL;
  PCHK(p, hipStreamSynchronize(p->st));
  return MAV1HIP_OK;
}

}  // extern "C"
