/* Motion search on gfx950: quarter-pel / decimated plane build and the
 * 4-level node search of the mav1 encoder (behaviour of
 * src/kernels/k_me.h:343-379 per node, src/backend_cpu.c:23-56 per frame).
 *
 * Plane build: one workgroup per 64 x 16 tile of a reference; the 23 x 71
 * source window (8-tap support, edge-clamped) is staged in LDS, the three
 * non-trivial horizontal phases are filtered once per row into LDS, and
 * each thread produces 4 adjacent pixels of all 16 phase planes.
 *
 * Node search: one workgroup per (node, reference). A few lanes share a
 * full-pel candidate, scored against the source block and the +-range search
 * window staged in LDS (edge clamping applied while staging, which
 * reproduces the per-coordinate clamping of the serial search); the winner is
 * the lexicographic minimum of (cost, candidate index), i.e. the serial
 * loop's first minimum. Sub-pel steps spread the 4x4 units of all of a ring's
 * candidates over the lanes; candidates are compared in ring order with a
 * strict <, as the serial refinement does.
 * Levels depend on their parent level and run as separate launches.
 */
#include "dev_common.h"
#include "internal.h"

#define TB(fp, bit) (((fp).turbo & (bit)) != 0)

long me_entry_bytes(const Mav1FrameParams &fp) {
  long W = fp.frame_w, H = fp.frame_h;
  return 16 * W * H + ((W + 3) >> 2) * ((H + 3) >> 2);
}
size_t me_dec_bytes(const Mav1FrameParams &fp) {
  return (size_t)((fp.frame_w + 3) >> 2) * ((fp.frame_h + 3) >> 2);
}

/* ------------------------------------------------------------------------ */
/* Quarter-pel planes                                                        */
/* ------------------------------------------------------------------------ */
#define QT_W 64
#define QT_H 16

DEVI void qpel_build_body(const Mav1FrameParams &fp, const uint8_t *__restrict__ ref, uint8_t *__restrict__ out, const int blk_x, const int blk_y, const int blk_z) {
  __shared__ uint8_t tile[QT_H + 7][QT_W + 8];
  __shared__ int16_t hz[3][QT_H + 7][QT_W];
  const int W = fp.frame_w, H = fp.frame_h, S = fp.stride[0];
  const uint8_t *luma = ref + fp.offset[0];
  const int x0 = blk_x * QT_W, y0 = blk_y * QT_H, tid = threadIdx.x;
  for (int i = tid; i < (QT_H + 7) * (QT_W + 7); i += 256) {
    int r = i / (QT_W + 7), c = i - r * (QT_W + 7);
    tile[r][c] = luma[d_clip(0, H - 1, y0 + r - 3) * S + d_clip(0, W - 1, x0 + c - 3)];
  }
  int kf[4][8];
#pragma unroll
  for (int f = 0; f < 4; f++)
#pragma unroll
    for (int t = 0; t < 8; t++) kf[f][t] = SUBPEL_FILTER(EIGHTTAP, 4 * f)[t];
  __syncthreads();
  /* horizontal phases 1..3 (phase 0 is the sample itself: Round2(128 p, 3) = 16 p) */
  for (int i = tid; i < (QT_H + 7) * QT_W; i += 256) {
    int r = i / QT_W, c = i - r * QT_W;
#pragma unroll
    for (int fx = 1; fx < 4; fx++) {
      int acc = 0;
#pragma unroll
      for (int u = 0; u < 8; u++) acc += kf[fx][u] * tile[r][c + u];
      hz[fx - 1][r][c] = (int16_t)d_round2(acc, 3);
    }
  }
  __syncthreads();
  const int tx = tid & 15, ty = tid >> 4;
  const int y = y0 + ty, xb = x0 + tx * 4;
  if (y >= H || xb >= W) return;
  const size_t n = (size_t)W * H, o = (size_t)y * W + xb;
  const bool wide = ((W & 3) == 0) && xb + 4 <= W;
#pragma unroll
  for (int fx = 0; fx < 4; fx++) {
    uint32_t word[4] = {0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < 4; p++) {
      int c = tx * 4 + p, col[8];
#pragma unroll
      for (int t = 0; t < 8; t++) col[t] = fx ? (int)hz[fx - 1][ty + t][c] : 16 * (int)tile[ty + t][c + 3];
#pragma unroll
      for (int fy = 0; fy < 4; fy++) {
        int acc = 0;
#pragma unroll
        for (int t = 0; t < 8; t++) acc += kf[fy][t] * col[t];
        word[fy] |= (uint32_t)d_clip1(d_round2(acc, 11)) << (8 * p);
      }
    }
#pragma unroll
    for (int fy = 0; fy < 4; fy++) {
      uint8_t *dst = out + (size_t)(fy * 4 + fx) * n + o;
      if (wide) {
        *(uint32_t *)dst = word[fy];
      } else {
        for (int p = 0; p < 4 && xb + p < W; p++) dst[p] = (uint8_t)(word[fy] >> (8 * p));
      }
    }
  }
}
__global__ __launch_bounds__(256) void k_qpel_build(const Mav1FrameParams fp, const uint8_t *__restrict__ ref,
                                                    uint8_t *__restrict__ out) {
  qpel_build_body(fp, ref, out, blockIdx.x, blockIdx.y, blockIdx.z);
}

hipError_t launch_qpel_build(hipStream_t st, const Mav1FrameParams &fp, const uint8_t *ref, uint8_t *planes16) {
  dim3 grid((fp.frame_w + QT_W - 1) / QT_W, (fp.frame_h + QT_H - 1) / QT_H);
  hipLaunchKernelGGL(k_qpel_build, grid, dim3(256), 0, st, fp, ref, planes16);
  return hipGetLastError();
}

/* 4x4-mean decimated plane (k_me.h:112-118 per sample). */
DEVI void dec_build_body(const Mav1FrameParams &fp, const uint8_t *__restrict__ frame, uint8_t *__restrict__ dec, const int blk_x, const int blk_y, const int blk_z) {
  const int W = fp.frame_w, H = fp.frame_h, dw = (W + 3) >> 2, dh = (H + 3) >> 2;
  const int x = blk_x * 64 + (threadIdx.x & 63), y = blk_y * 4 + (threadIdx.x >> 6);
  if (x >= dw || y >= dh) return;
  const uint8_t *luma = frame + fp.offset[0];
  int s = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint8_t *row = luma + d_clip(0, H - 1, 4 * y + i) * fp.stride[0];
#pragma unroll
    for (int j = 0; j < 4; j++) s += row[d_clip(0, W - 1, 4 * x + j)];
  }
  dec[(size_t)y * dw + x] = (uint8_t)((s + 8) >> 4);
}
__global__ __launch_bounds__(256) void k_dec_build(const Mav1FrameParams fp, const uint8_t *__restrict__ frame,
                                                   uint8_t *__restrict__ dec) {
  dec_build_body(fp, frame, dec, blockIdx.x, blockIdx.y, blockIdx.z);
}

hipError_t launch_dec_build(hipStream_t st, const Mav1FrameParams &fp, const uint8_t *frame, uint8_t *dec) {
  int dw = (fp.frame_w + 3) >> 2, dh = (fp.frame_h + 3) >> 2;
  hipLaunchKernelGGL(k_dec_build, dim3((dw + 63) / 64, (dh + 3) / 4), dim3(256), 0, st, fp, frame, dec);
  return hipGetLastError();
}

/* ------------------------------------------------------------------------ */
/* Node search                                                               */
/* ------------------------------------------------------------------------ */
/* Threads of a node's workgroup and, in the full-pel stages, the lanes that
 * share a candidate (each takes every ME_G-th row): many for the few large
 * nodes, whose 50 to 290 candidates of up to 4096 samples are a node's
 * latency; one wave for the 16x16 and 8x8 nodes, which fill the chip. */
template <int LEVEL>
constexpr int ME_NT = LEVEL == 0 ? 512 : LEVEL == 1 ? 256 : 64;
template <int LEVEL>
constexpr int ME_G = LEVEL <= 1 ? 8 : 2;
/* Largest full-pel radius served from the LDS window. */
template <int LEVEL>
constexpr int ME_WIN = LEVEL == 0 ? 32 : 4;
#define ME_DEC_R 8 /* largest radius of the decimated window (full-pel radius 32) */

struct NodeState {
  int x, y, cy, cx, range, step, nstage, pr, pc, copy, valid;
};

DEVI void me_cand(const NodeState &m, int k, int &dy, int &dx) {
  if (k == 0) {
    dy = m.cy;
    dx = m.cx;
    return;
  }
  int side = 2 * (m.range / m.step) + 1;
  int q = (k - 1) / side;
  dy = m.cy - m.range + q * m.step;
  dx = m.cx - m.range + (k - 1 - q * side) * m.step;
}

DEVI int me_bits(int dy, int dx) {
  return 2 + 2 * d_floorlog2((unsigned)(d_abs(dy) * 8 + 1)) + 2 * d_floorlog2((unsigned)(d_abs(dx) * 8 + 1));
}

typedef __attribute__((address_space(3))) const uint32_t lds_cu32;
/* Byte `at` on of an LDS array of words, as words. */
struct LdsBytes {
  const lds_cu32 *p;
  uint32_t w;
  int s;
  DEVI LdsBytes(const uint8_t *base, int at) {
    p = (const lds_cu32 *)(base + (at & ~3));
    s = at & 3;
    w = *p++;
  }
  DEVI uint32_t next() {
    const uint32_t n = *p++, v = __builtin_amdgcn_alignbyte(n, w, s);
    w = n;
    return v;
  }
};
/* SAD of rows first, + stride, .. of an N x N block at srcL (row stride N)
 * against the window (row stride WS) from (oy, ox) on. */
template <int N, int WS>
DEVI int sad_rows(const uint8_t *srcL, const uint8_t *win, int oy, int ox, int first, int stride) {
  uint32_t s = 0;
  for (int i = first; i < N; i += stride) {
    const lds_cu32 *a = (const lds_cu32 *)(srcL + i * N);
    LdsBytes b(win, (i + oy) * WS + ox);
#pragma unroll
    for (int j = 0; j < N / 4; j++) s = __builtin_amdgcn_sad_u8(a[j], b.next(), s);
  }
  return (int)s;
}
/* The same against the frame (coordinates clamped), for radii past the window. */
template <int BW>
DEVI int sad_rows_global(const Mav1FrameParams &fp, const uint8_t *srcL, const uint8_t *refY, int x, int y, int dy,
                         int dx, int first, int stride) {
  int s = 0, S = fp.stride[0];
  for (int i = first; i < BW; i += stride) {
    const uint8_t *b = refY + d_clip(0, fp.frame_h - 1, y + i + dy) * S;
    for (int j = 0; j < BW; j++) s += d_abs((int)srcL[i * BW + j] - (int)b[d_clip(0, fp.frame_w - 1, x + j + dx)]);
  }
  return s;
}
template <int BW>
DEVI int sad_rows_dec_global(const Mav1FrameParams &fp, const uint8_t *ds, const uint8_t *dr, int x, int y, int dy,
                             int dx, int first, int stride) {
  const int W = (fp.frame_w + 3) >> 2, H = (fp.frame_h + 3) >> 2, n = BW >> 2;
  const int x0 = x >> 2, y0 = y >> 2, oy = dy >> 2, ox = dx >> 2;
  int s = 0;
  for (int i = first; i < n; i += stride) {
    const uint8_t *a = ds + d_min(y0 + i, H - 1) * W, *b = dr + d_clip(0, H - 1, y0 + i + oy) * W;
    for (int j = 0; j < n; j++) s += d_abs((int)a[d_min(x0 + j, W - 1)] - (int)b[d_clip(0, W - 1, x0 + j + ox)]);
  }
  return s;
}
/* Sum over the G lanes that share a candidate (in every one of them). */
template <int G>
DEVI int me_group_sum(int v) {
  v += dpp_t<DPP_QX1>(v);
  if constexpr (G == 8) {
    v += dpp_t<DPP_QX2>(v);
    v += dpp_t<DPP_HMIRROR>(v);
  }
  return v;
}

/* The normative EIGHTTAP prediction (7.11.3) of a 4x4 unit at an even
 * 1/8-pel vector, from the staged window: (wy, wx) the window position of the
 * unit's first sample, phases fy, fx in quarter samples. d: source minus
 * prediction. The horizontal taps are signed bytes times (sample - 128) on
 * the dot products (the whole-sample phase's 128 as 2 * 64), the vertical
 * ones pairs of 16 bits. */
struct MeTaps {
  uint32_t h[4][2], v[4][4];
};
DEVI void me_taps(MeTaps &T, int tid) {
  if (tid < 4) {
    const int16_t *k = SUBPEL_FILTER(EIGHTTAP, 4 * tid);
    uint32_t w[2] = {0, 0};
    for (int t = 0; t < 8; t++) {
      w[t >> 2] |= (uint32_t)((tid ? k[t] : k[t] / 2) & 255) << (8 * (t & 3));
      if (!(t & 1)) T.v[tid][t >> 1] = (uint32_t)(k[t] & 0xFFFF) | (uint32_t)(k[t + 1] & 0xFFFF) << 16;
    }
    T.h[tid][0] = w[0];
    T.h[tid][1] = w[1];
  }
}
template <int WS>
DEVI void me_pred_diff(const MeTaps &T, const uint8_t *win, int wy, int wx, int fy, int fx, const uint32_t src[4],
                       int d[16]) {
  typedef short s2 __attribute__((ext_vector_type(2)));
  union P {
    uint32_t u;
    s2 v;
  };
  const int t0 = (int)T.h[fx][0], t1 = (int)T.h[fx][1], sh = fx ? 0 : 1;
  int m[4][11];
#pragma unroll
  for (int r = 0; r < 11; r++) {
    LdsBytes b(win, (wy - 3 + r) * WS + wx - 3);
    const uint32_t n0 = b.next() ^ 0x80808080u, n1 = b.next() ^ 0x80808080u, n2 = b.next() ^ 0x80808080u;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int lo = (int)__builtin_amdgcn_alignbyte(n1, n0, j), hi = (int)__builtin_amdgcn_alignbyte(n2, n1, j);
      const int a = __builtin_amdgcn_sdot4(hi, t1, __builtin_amdgcn_sdot4(lo, t0, 0, false), false);
      m[j][r] = ((a << sh) + 16384 + 4) >> 3;
    }
  }
  P v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) v[i].u = T.v[fy][i];
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
      d[4 * i + j] = (int)((src[i] >> (8 * j)) & 255) - d_clip1(a >> 11);
    }
  }
}

/* HP: sub-pel costs from the quarter-pel planes, else from predictions.
 * One workgroup per (node, reference). Full-pel stages: ME_G lanes share a
 * candidate, four samples per instruction, source, window and the decimated
 * planes' windows staged in LDS. Sub-pel rings: a ring's candidates do not
 * depend on each other, so the lanes take (candidate, 4x4 unit) pairs of the
 * whole ring and the serial walk over the costs keeps its first minimum.
 * Bound by the latency of the stages at small frames and by LDS reads and
 * VALU issue at large ones. Levels 0 .. 3 at 352x288: 18, 7, 13 and 8 us
 * (turbo), 58, 18, 25 and 22 us (full search); with one wave per node, a lane
 * per candidate, byte loads and one prediction after another 100, 25, 19 and
 * 10 us, 811, 123, 64 and 80 us. */
template <int LEVEL, bool HP>
DEVI void me_level_body(const Mav1FrameParams &fp, const uint8_t *__restrict__ src, const uint8_t *__restrict__ ref0, const uint8_t *__restrict__ ref1, const uint8_t *__restrict__ planes, long entryBytes, const uint8_t *__restrict__ srcDec, int32_t *__restrict__ field0, int32_t *__restrict__ field1, int nodesPerRef, const int blk_x, const int blk_y, const int blk_z) {
  constexpr int BW = 64 >> LEVEL, NT = ME_NT<LEVEL>, NW = NT / 64, G = ME_G<LEVEL>, R = ME_WIN<LEVEL>;
  constexpr int N = 1 << LEVEL;
  constexpr int WR = BW + (2 * R > 9 ? 2 * R : 9); /* window rows: full-pel radius R, or the predictions' support */
  constexpr int WS = ((WR + 3) & ~3) + 4;          /* row stride: words, one more to read ahead */
  constexpr int DN = BW / 4, DR = DN + 2 * ME_DEC_R, DS = ((DR + 3) & ~3) + 4;
  __shared__ alignas(16) uint8_t srcL[BW * BW];
  __shared__ alignas(16) uint8_t win[WR * WS + 16];
  __shared__ alignas(16) uint8_t dsrc[LEVEL ? 4 : DN * DN], dwin[LEVEL ? 4 : DR * DS + 16];
  __shared__ MeTaps taps;
  __shared__ unsigned long long smin[2][NW];
  __shared__ int scost[2][9];
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = blk_x / nodesPerRef, node = blk_x - r * nodesPerRef;
  const int sb = node >> (2 * LEVEL), i = node & (N * N - 1);
  const uint8_t *ref = r ? ref1 : ref0;
  int32_t *field = r ? field1 : field0;
  const uint8_t *pl = planes + r * entryBytes;
  const uint8_t *refDec = pl + (size_t)16 * fp.frame_w * fp.frame_h;

  NodeState m;
  m.x = (sb % fp.sb_cols) * 64 + (i % N) * BW;
  m.y = (sb / fp.sb_cols) * 64 + (i / N) * BW;
  int32_t *out = field + (sb * MAV1_NUM_NODES + d_node_base(LEVEL) + i) * 2;
  if (m.x >= fp.frame_w || m.y >= fp.frame_h) {
    if (tid == 0) out[0] = out[1] = 0;
    return;
  }
  m.range = fp.me_range;
  m.step = 1;
  m.nstage = 1;
  m.pr = m.pc = m.cy = m.cx = 0;
  m.copy = 0;
  if (LEVEL > 0) {
    int parent = ((i / N) >> 1) * (N >> 1) + ((i % N) >> 1);
    const int32_t *pv = field + (sb * MAV1_NUM_NODES + d_node_base(LEVEL - 1) + parent) * 2;
    m.pr = pv[0];
    m.pc = pv[1];
    m.cy = m.pr >> 3;
    m.cx = m.pc >> 3;
    m.range = d_min(m.range, TB(fp, MAV1_T_ME_CR1) ? 1 : TB(fp, MAV1_T_ME_CR2) ? 2 : 4);
    bool leafNo8 = TB(fp, MAV1_T_LEAF_NO8) && fp.leaf && !fp.frame_is_intra;
    m.copy = LEVEL == 3 && (TB(fp, MAV1_T_ME_L3COPY) || leafNo8);
  } else {
    m.step = TB(fp, MAV1_T_ME_HME3) ? 8 : 4;
    m.range = (m.range / m.step) * m.step;
    m.nstage = TB(fp, MAV1_T_ME_HME3) ? 3 : 2;
  }
  if (LEVEL == 3 && TB(fp, MAV1_T_ME_L3SUB)) m.nstage = 0;
  if (r && LEVEL == 3 && TB(fp, MAV1_T_ME_G3COPY) && fp.leaf && !fp.frame_is_intra) m.copy = 1;
  if (m.copy) {
    if (tid == 0) {
      out[0] = m.pr;
      out[1] = m.pc;
    }
    return;
  }
  const int S = fp.stride[0], H1 = fp.frame_h - 1, W1 = fp.frame_w - 1;
  const uint8_t *srcY = src + fp.offset[0], *refY = ref + fp.offset[0];
#pragma unroll
  for (int k = 0; k < BW * BW / NT; k++) {
    const int q = tid + k * NT;
    srcL[q] = srcY[(m.y + q / BW) * S + m.x + (q % BW)];
  }
  if constexpr (!HP) me_taps(taps, tid);
  /* the reference around (y, x) into the window: rows x cols samples, clamped */
  auto stage = [&](int y, int x, int n) {
    const int c0 = tid & 63;
    for (int wr = tid >> 6; wr < n; wr += NW)
      for (int wc = c0; wc < n; wc += 64) win[wr * WS + wc] = refY[d_clip(0, H1, y + wr) * S + d_clip(0, W1, x + wc)];
  };

  int by = 0, bx = 0;
  for (int stg = 0; stg < m.nstage; stg++) {
    if (stg > 0) {
      m.cy = by;
      m.cx = bx;
      if (stg == 1 && TB(fp, MAV1_T_ME_HME3)) {
        m.range = 4;
        m.step = 4;
      } else {
        m.range = TB(fp, MAV1_T_ME_REF2) ? 2 : 3;
        m.step = 1;
      }
    }
    const int side = 2 * (m.range / m.step) + 1, count = 1 + side * side;
    const bool dec = TB(fp, MAV1_T_ME_DEC) && m.step >= 4;
    const int rs = (TB(fp, MAV1_T_ME_RSUB) && m.step == 1) ? 2 : 1;
    const bool lds = m.range <= (dec ? (LEVEL ? -1 : 4 * ME_DEC_R) : R);
    const int oy0 = m.cy - m.range, ox0 = m.cx - m.range;
    if (stg) __syncthreads(); /* the last stage's reads of the windows */
    if constexpr (LEVEL == 0) {
      if (dec && lds) {
        const int W = (fp.frame_w + 3) >> 2, H = (fp.frame_h + 3) >> 2, x0 = m.x >> 2, y0 = m.y >> 2;
        const int oy = oy0 >> 2, ox = ox0 >> 2, n = DN + 2 * (m.range >> 2);
        if (tid < DN * DN) dsrc[tid] = srcDec[(size_t)d_min(y0 + tid / DN, H - 1) * W + d_min(x0 + tid % DN, W - 1)];
        for (int wr = tid >> 5; wr < n; wr += NT / 32) /* n <= 32 */
          if ((tid & 31) < n)
            dwin[wr * DS + (tid & 31)] =
                refDec[(size_t)d_clip(0, H - 1, y0 + oy + wr) * W + d_clip(0, W - 1, x0 + ox + (tid & 31))];
      }
    }
    if (!dec && lds) stage(m.y + oy0, m.x + ox0, BW + 2 * m.range);
    __syncthreads();
    unsigned long long best = ~0ull;
    const int g = tid & (G - 1);
    for (int k = tid / G; k < ((count + NT / G - 1) & ~(NT / G - 1)); k += NT / G) {
      int dy, dx;
      const int kk = d_min(k, count - 1);
      me_cand(m, kk, dy, dx);
      const int rate = fp.ac_q[0] * me_bits(dy, dx) / 64;
      int c;
      if (dec) {
        if (LEVEL == 0 && lds)
          c = sad_rows<DN, DS>(dsrc, dwin, (dy - oy0) >> 2, (dx - ox0) >> 2, g, G);
        else
          c = sad_rows_dec_global<BW>(fp, srcDec, refDec, m.x, m.y, dy, dx, g, G);
        c *= 16;
      } else if (lds) {
        c = sad_rows<BW, WS>(srcL, win, dy - oy0, dx - ox0, g * rs, G * rs) * rs;
      } else {
        c = sad_rows_global<BW>(fp, srcL, refY, m.x, m.y, dy, dx, g * rs, G * rs) * rs;
      }
      const unsigned long long key = pack_key(me_group_sum<G>(c) + rate, kk);
      best = key < best ? key : best;
    }
    best = wave_min_u64(best);
    if constexpr (NW > 1) {
      if (lane == 0) smin[stg & 1][tid >> 6] = best;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < NW; w++) best = smin[stg & 1][w] < best ? smin[stg & 1][w] : best;
    }
    me_cand(m, (int)(best & 0xffffffffu), by, bx);
  }
  if (LEVEL > 0 && TB(fp, MAV1_T_ME_KEEP) && by == m.cy && bx == m.cx) {
    if (tid == 0) {
      out[0] = m.pr;
      out[1] = m.pc;
    }
    return;
  }
  /* sub-pel refinement: half-pel ring, then quarter-pel ring unless
   * T_ME_HALF01 stops nodes >= 32 wide at half-pel */
  int mvr = m.nstage ? by * 8 : m.pr, mvc = m.nstage ? bx * 8 : m.pc;
  constexpr int NR = BW / 4;
  const int st = (HP && TB(fp, MAV1_T_ME_USUB) && BW >= 32) ? 2 : 1, nue = NR * NR / st;
  const int minStep = (BW >= 32 && TB(fp, MAV1_T_ME_HALF01)) ? 4 : 2;
  const bool cross = TB(fp, MAV1_T_ME_CROSS);
  /* the predictions' support around every vector the two rings can reach */
  const int wy0 = ((mvr - 6) >> 3) - 3, wx0 = ((mvc - 6) >> 3) - 3;
  if constexpr (!HP) {
    __syncthreads();
    stage(m.y + wy0, m.x + wx0, BW + 9);
  }
  int bestS = 0;
  for (int step = 4; step >= minStep; step >>= 1) {
    const int cr0 = mvr, cc0 = mvc, first = step == 4, ring = cross ? 4 : 8, n = first + ring;
    /* candidate k: the centre (first ring), then the ring in its order */
    auto vec = [&](int k, int &vr, int &vc) {
      const int q = k - first, j = cross ? (q == 0 ? 1 : q == 1 ? 3 : q == 2 ? 4 : 6) : q;
      vr = cr0 + (q < 0 ? 0 : j < 3 ? -1 : j < 5 ? 0 : 1) * step;
      vc = cc0 + (q < 0 ? 0 : (j == 0 || j == 3 || j == 5) ? -1 : (j == 1 || j == 6) ? 0 : 1) * step;
    };
    int *cost = scost[first];
    if (tid < n) cost[tid] = 0;
    __syncthreads();
    for (int p = tid; p < n * nue; p += NT) {
      const int c = p / nue, u = (p - c * nue) * st;
      int vr, vc;
      vec(c, vr, vc);
      const int ucol = u % NR, urow = u / NR;
      uint32_t sw[4];
#pragma unroll
      for (int q = 0; q < 4; q++) sw[q] = *(const lds_cu32 *)(srcL + (urow * 4 + q) * BW + ucol * 4);
      int d[16];
      if constexpr (HP) {
        const int W = fp.frame_w, iy = m.y + urow * 4 + (vr >> 3), ix = m.x + ucol * 4 + (vc >> 3);
        const uint8_t *base = pl + (size_t)(((vr >> 1) & 3) * 4 + ((vc >> 1) & 3)) * W * fp.frame_h;
        uint32_t pw[4];
        if (ix >= 0 && ix + 3 < W) {
#pragma unroll
          for (int q = 0; q < 4; q++) __builtin_memcpy(&pw[q], base + (size_t)d_clip(0, H1, iy + q) * W + ix, 4);
        } else {
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const uint8_t *prow = base + (size_t)d_clip(0, H1, iy + q) * W;
            pw[q] = prow[d_clip(0, W1, ix)] | (uint32_t)prow[d_clip(0, W1, ix + 1)] << 8 |
                    (uint32_t)prow[d_clip(0, W1, ix + 2)] << 16 | (uint32_t)prow[d_clip(0, W1, ix + 3)] << 24;
          }
        }
#pragma unroll
        for (int q = 0; q < 16; q++)
          d[q] = (int)((sw[q >> 2] >> (8 * (q & 3))) & 255) - (int)((pw[q >> 2] >> (8 * (q & 3))) & 255);
      } else {
        me_pred_diff<WS>(taps, win, urow * 4 + (vr >> 3) - wy0, ucol * 4 + (vc >> 3) - wx0, (vr >> 1) & 3, (vc >> 1) & 3,
                         sw, d);
      }
      /* the lanes of a quad or a row of 16 have the same candidate */
      int s = satd4x4_arr(d) * st;
      s += dpp_t<DPP_QX1>(s);
      s += dpp_t<DPP_QX2>(s);
      if constexpr (BW >= 16) {
        s += dpp_t<DPP_HMIRROR>(s);
        s += dpp_t<DPP_MIRROR>(s);
        if ((lane & 15) == 0) atomicAdd(&cost[c], s);
      } else {
        if ((lane & 3) == 0) atomicAdd(&cost[c], s);
      }
    }
    __syncthreads();
    if (first) bestS = cost[0];
    for (int k = first; k < n; k++) {
      const int c = cost[k];
      if (c < bestS) {
        bestS = c;
        vec(k, mvr, mvc);
      }
    }
  }
  if (tid == 0) {
    out[0] = mvr;
    out[1] = mvc;
  }
}
template <int LEVEL, bool HP>
__global__ __launch_bounds__(ME_NT<LEVEL>) void k_me_level(const Mav1FrameParams fp, const uint8_t *__restrict__ src,
                                                 const uint8_t *__restrict__ ref0, const uint8_t *__restrict__ ref1,
                                                 const uint8_t *__restrict__ planes, long entryBytes,
                                                 const uint8_t *__restrict__ srcDec, int32_t *__restrict__ field0,
                                                 int32_t *__restrict__ field1, int nodesPerRef) {
  me_level_body<LEVEL, HP>(fp, src, ref0, ref1, planes, entryBytes, srcDec, field0, field1, nodesPerRef,
                           xcd_item(blockIdx.x, gridDim.x, 1 << (2 * LEVEL)), blockIdx.y, blockIdx.z);
}

template <int LEVEL>
static void launch_level(hipStream_t st, bool hp, dim3 grid, const Mav1FrameParams &fp, const uint8_t *src,
                         const uint8_t *ref0, const uint8_t *ref1, const uint8_t *planes, long entryBytes,
                         const uint8_t *srcDec, int32_t *field0, int32_t *field1, int nodesPerRef) {
  if (hp)
    hipLaunchKernelGGL((k_me_level<LEVEL, true>), grid, dim3(ME_NT<LEVEL>), 0, st, fp, src, ref0, ref1, planes, entryBytes, srcDec,
                       field0, field1, nodesPerRef);
  else
    hipLaunchKernelGGL((k_me_level<LEVEL, false>), grid, dim3(ME_NT<LEVEL>), 0, st, fp, src, ref0, ref1, planes, entryBytes,
                       srcDec, field0, field1, nodesPerRef);
}

hipError_t launch_me_level(hipStream_t st, int level, const Mav1FrameParams &fp, const uint8_t *src,
                           const uint8_t *ref0, const uint8_t *ref1, const uint8_t *planes, long entryBytes,
                           const uint8_t *srcDec, int32_t *field0, int32_t *field1, int nref) {
  int nodesPerRef = fp.sb_cols * fp.sb_rows << (2 * level);
  dim3 grid(nodesPerRef * nref);
  const bool hp = (fp.turbo & MAV1_T_ME_HPEL) != 0;
  switch (level) {
    case 0: launch_level<0>(st, hp, grid, fp, src, ref0, ref1, planes, entryBytes, srcDec, field0, field1, nodesPerRef); break;
    case 1: launch_level<1>(st, hp, grid, fp, src, ref0, ref1, planes, entryBytes, srcDec, field0, field1, nodesPerRef); break;
    case 2: launch_level<2>(st, hp, grid, fp, src, ref0, ref1, planes, entryBytes, srcDec, field0, field1, nodesPerRef); break;
    default: launch_level<3>(st, hp, grid, fp, src, ref0, ref1, planes, entryBytes, srcDec, field0, field1, nodesPerRef); break;
  }
  return hipGetLastError();
}

/* ---- batched launches (batch.h): the same kernels over several frames ---- */

/* which 0: LAST's planes, 1: the second reference's. */
__global__ __launch_bounds__(256) void k_qpel_build_b(const BatchFrame *__restrict__ T, const BatchGrid g, int which) {
  const BatchIdx b = batch_idx(g);
  const BatchFrame &F = T[b.f];
  qpel_build_body(F.fp, which ? gptr(F.gold) : gptr(F.ref), gptr(F.planes) + which * F.entry_bytes, b.x, b.y, b.z);
}

hipError_t launch_qpel_build_b(hipStream_t st, const BatchFrame *T, const BatchFrame *H, int n, int which) {
  BatchGrid g = batch_grid();
  for (int f = 0; f < n; f++)
    batch_grid_add(g, (H[f].fp.frame_w + QT_W - 1) / QT_W, (H[f].fp.frame_h + QT_H - 1) / QT_H, 1);
  hipLaunchKernelGGL(k_qpel_build_b, dim3(g.start[n]), dim3(256), 0, st, T, g, which);
  return hipGetLastError();
}

/* which 0 / 1: the decimated plane of LAST / the second reference behind
 * its 16 quarter-pel planes; 2: the source's, after both entries. */
__global__ __launch_bounds__(256) void k_dec_build_b(const BatchFrame *__restrict__ T, const BatchGrid g, int which) {
  const BatchIdx b = batch_idx(g);
  const BatchFrame &F = T[b.f];
  const size_t n16 = (size_t)16 * F.fp.frame_w * F.fp.frame_h;
  const uint8_t *frame = which == 2 ? gptr(F.src) : which ? gptr(F.gold) : gptr(F.ref);
  uint8_t *dec = which == 2 ? gptr(F.planes) + 2 * F.entry_bytes : gptr(F.planes) + which * F.entry_bytes + n16;
  dec_build_body(F.fp, frame, dec, b.x, b.y, b.z);
}

hipError_t launch_dec_build_b(hipStream_t st, const BatchFrame *T, const BatchFrame *H, int n, int which) {
  BatchGrid g = batch_grid();
  for (int f = 0; f < n; f++) {
    const int dw = (H[f].fp.frame_w + 3) >> 2, dh = (H[f].fp.frame_h + 3) >> 2;
    batch_grid_add(g, (dw + 63) / 64, (dh + 3) / 4, 1);
  }
  hipLaunchKernelGGL(k_dec_build_b, dim3(g.start[n]), dim3(256), 0, st, T, g, which);
  return hipGetLastError();
}

template <int LEVEL, bool HP>
__global__ __launch_bounds__(ME_NT<LEVEL>) void k_me_level_b(const BatchFrame *__restrict__ T, const BatchGrid g) {
  const BatchIdx b = batch_idx(g, xcd_item(blockIdx.x, gridDim.x, 1 << (2 * LEVEL)));
  const BatchFrame &F = T[b.f];
  me_level_body<LEVEL, HP>(F.fp, gptr(F.src), gptr(F.ref), gptr(F.gold), gptr(F.planes), (long)F.entry_bytes, gptr(F.planes) + 2 * F.entry_bytes,
                           gptr(F.mvf), gptr(F.mvg), g.aux[b.f], b.x, b.y, b.z);
}

template <int LEVEL>
static void launch_level_b(hipStream_t st, bool hp, const BatchFrame *T, const BatchGrid &g) {
  if (hp)
    hipLaunchKernelGGL((k_me_level_b<LEVEL, true>), dim3(g.start[g.n]), dim3(ME_NT<LEVEL>), 0, st, T, g);
  else
    hipLaunchKernelGGL((k_me_level_b<LEVEL, false>), dim3(g.start[g.n]), dim3(ME_NT<LEVEL>), 0, st, T, g);
}

hipError_t launch_me_level_b(hipStream_t st, int level, const BatchFrame *T, const BatchFrame *H, int n, int nref) {
  BatchGrid g = batch_grid();
  for (int f = 0; f < n; f++) {
    const int nodesPerRef = H[f].fp.sb_cols * H[f].fp.sb_rows << (2 * level);
    batch_grid_add(g, nodesPerRef * nref, 1, 1, nodesPerRef);
  }
  const bool hp = (H[0].fp.turbo & MAV1_T_ME_HPEL) != 0;
  switch (level) {
    case 0: launch_level_b<0>(st, hp, T, g); break;
    case 1: launch_level_b<1>(st, hp, T, g); break;
    case 2: launch_level_b<2>(st, hp, T, g); break;
    default: launch_level_b<3>(st, hp, T, g); break;
  }
  return hipGetLastError();
}
