// q3h_gemm.hip - the int8 path of the Q8_0 products (stacks created with
// act_q8 = 1): activations are quantized per 32-block with the weights' own
// quantizer (ggml quantize_row_q8_0_ref: d = amax / 127, q = round(x / d)
// half away from zero, d kept as fp16; the format of lm.pas:259-267), then
// every Q8_0 block of the product is one v_mfma_i32_16x16x32_i8 whose exact
// int32 dot is scaled by d_w * d_x into an fp32 sum (ggml
// vec_dot_q8_0_q8_0).
//
// Evaluation order (fixed, so that the products equal a CPU evaluation in the
// same order to the bit): per output, one fused multiply-add chain over the
// 16 blocks of each 512-column chunk, acc = fma((float)dot_b, d_w * d_x, acc)
// from 0 in block order, and the chunk sums added in chunk order.
//
// Operand layouts (v_mfma_i32_16x16x32_i8, wave64): lane l holds 8 int8 of
// row l % 16 of A and of column l % 16 of B, k = 8 * (l / 16) .. + 7; the
// result C[4 * (l / 16) + r][l % 16], r < 4, lands in lane l. A is 16 weight
// rows, B 16 activation rows, both stored in operand order (launch_tile_q8: the
// matrices of an act_q8 stack are rewritten so at load; qtile_offset: written
// so by the quantizers), so one coalesced 1 KB load gives the operands of two
// blocks.
//
// Three schedules of the same chains:
//  - k_gemm_i8: a workgroup per 16 weight rows, its waves taking the chunks
//    and adding them through LDS; any number of rows (prefill);
//  - k_gemm_i8r: a wave per 64 weight rows and activation tile over the whole
//    K, where these fill the chip (long or several prompts);
//  - k_gemm_i8p (up to 64 rows, the batched decode step): one wave per (16
//    weight rows, chunk) over the whole chip, the chunk sums written out as
//    partials that the consumer adds in chunk order (k_quant_act with a
//    partial source, or the attention prologue).
#include "q3h_internal.h"
#include "q3h_math.h"
#include "q3h_wave.h"

namespace q3h {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kQuantThreads = 128;
constexpr int kQuantChunks = 3;  // 8-element chunks per thread: K <= 3072
constexpr int kChunkBlocks = 16;  // 32-blocks per chunk of a product (512 columns)
constexpr int kMaxChunks = 6;     // chunks of a product: K <= 3072

__device__ __forceinline__ float *scales_of(int8_t *xq, int M, int K) {
  return reinterpret_cast<float *>(xq + (size_t)((M + 15) & ~15) * K);
}

// block h (0, 1) of a lane's 16 operand bytes of a pair of blocks
__device__ __forceinline__ long half_pair(const int4 &v, int h) {
  return h ? ((long)(unsigned)v.w << 32) | (unsigned)v.z : ((long)(unsigned)v.y << 32) | (unsigned)v.x;
}

// The quantizer. One workgroup per activation row m < Mp and slice of its
// 8-element chunks (gridDim.x == Mp, M rounded up to 16; gridDim.y == nsl
// slices): a thread owns chunks j = blockIdx.y * 128 + t + i * 128 * nsl, and the
// four chunks of a lane quad make one 32-block. Rows M..Mp-1 are written as
// zeros. The row is
//  SRC_X:      x[m][0..K) (row stride ld);
//  SRC_ADD:    x[m] + sum_c part[c][m] (c < ld <= kMaxChunks chunk partials
//              of a product with N = K, added in chunk order), written back
//              to x (the residual stream, row stride K);
//  SRC_SWIGLU: silu(sum_c part[c][m][2k]) * sum_c part[c][m][2k + 1] (c < ld
//              <= 2 partials; gate / up interleaved, N = 2K).
// Then RMSNorm when norm_w != nullptr (one slice only): y = w * (x * inv),
// inv = 1/sqrt(mean(x^2) + eps) with the sum of squares in double; xn_out,
// when non-null, receives the (normed) rows M - xn_rows .. M - 1 (row
// M - xn_rows + r at xn_out + r K); and the Q8_0 blocks
// (skipped when xq == nullptr). Partial loads are all issued before the sums.
enum { SRC_X = 0, SRC_ADD = 1, SRC_SWIGLU = 2 };

// KC: chunks per thread (the row's chunks / (128 slices), rounded up); NC: the
// partial slots read (ld <= NC; SRC_ADD and SRC_SWIGLU). The arguments the
// loads depend on (the slice count among them, instead of gridDim) sit in the
// first 14 dwords, which arrive preloaded in SGPRs; xn_out, used only at the
// end, comes last.
template <int SRC, int KC, int NC>
__global__ __launch_bounds__(kQuantThreads) void k_quant_act(float *x, const float *part,
                                                              int8_t *xq, const float *norm_w,
                                                              int M, int K, int ld, float eps,
                                                              int nsl, float *xn_out,
                                                              int xn_rows) {
  const int m = blockIdx.x, t = threadIdx.x;
  const int mt16 = (M + 15) >> 4, nch = K >> 3, nb = K >> 5;
  const int j0 = blockIdx.y * kQuantThreads + t, js = kQuantThreads * nsl;
  float *dx = xq ? scales_of(xq, M, K) : nullptr;
  if (m >= M) {
    if (xq)
      for (int j = j0; j < nch; j += js) {
        *reinterpret_cast<long *>(xq + qtile_offset(m, 8 * j, mt16)) = 0;
        if ((j & 3) == 0) dx[qscale_offset(m, j >> 2, nb)] = 0.f;
      }
    return;
  }
  // the norm weights of this thread's chunks, loaded first (they are read by
  // every row, so they come from L2 before the partials arrive)
  float4 wpre[KC][2];
  if (norm_w) {
    const float4 *wr = reinterpret_cast<const float4 *>(norm_w);
#pragma unroll
    for (int i = 0; i < KC; i++) {
      const int jc = min(j0 + i * js, nch - 1);
      wpre[i][0] = wr[2 * jc];
      wpre[i][1] = wr[2 * jc + 1];
    }
  }
  // loads from clamped chunk / partial indices (a guarded load would be waited
  // for on its own); chunks past the row and partials past ld contribute zeros
  float v[KC][8];
#pragma unroll
  for (int i = 0; i < KC; i++) {
    const int j = j0 + i * js, jc = min(j, nch - 1);
    const bool on = j < nch;
    if (SRC == SRC_X) {
      const float4 *xr = reinterpret_cast<const float4 *>(x + (size_t)m * ld);
      const float4 a = xr[2 * jc], b = xr[2 * jc + 1];
      const float x8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int e = 0; e < 8; e++) v[i][e] = on ? x8[e] : 0.f;
    } else if (SRC == SRC_ADD) {
      float4 pa[NC], pb[NC];
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const float4 *pr =
            reinterpret_cast<const float4 *>(part + ((size_t)min(c, ld - 1) * M + m) * K);
        pa[c] = pr[2 * jc];
        pb[c] = pr[2 * jc + 1];
      }
      float4 *xr = reinterpret_cast<float4 *>(x + (size_t)m * K);
      const float4 a = xr[2 * jc], b = xr[2 * jc + 1];
      float s[8];
#pragma unroll
      for (int e = 0; e < 8; e++) s[e] = 0.f;
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const float p8[8] = {pa[c].x, pa[c].y, pa[c].z, pa[c].w,
                             pb[c].x, pb[c].y, pb[c].z, pb[c].w};
#pragma unroll
        for (int e = 0; e < 8; e++) s[e] = c < ld ? __fadd_rn(s[e], p8[e]) : s[e];
      }
      const float h8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int e = 0; e < 8; e++) v[i][e] = on ? __fadd_rn(h8[e], s[e]) : 0.f;
      if (on) {
        xr[2 * j] = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
        xr[2 * j + 1] = make_float4(v[i][4], v[i][5], v[i][6], v[i][7]);
      }
    } else {
      constexpr int MC = NC;
      float4 pr[MC][4];
#pragma unroll
      for (int c = 0; c < MC; c++) {
        const float4 *pp =
            reinterpret_cast<const float4 *>(part + ((size_t)min(c, ld - 1) * M + m) * (2 * K)) +
            4 * jc;
#pragma unroll
        for (int q = 0; q < 4; q++) pr[c][q] = pp[q];
      }
      float gs[8], us[8];
#pragma unroll
      for (int e = 0; e < 8; e++) gs[e] = us[e] = 0.f;
#pragma unroll
      for (int c = 0; c < MC; c++) {
        if (c >= ld) break;  // uniform
#pragma unroll
        for (int q = 0; q < 4; q++) {  // gate, up of outputs 8j + 2q, 8j + 2q + 1
          gs[2 * q] = __fadd_rn(gs[2 * q], pr[c][q].x);
          us[2 * q] = __fadd_rn(us[2 * q], pr[c][q].y);
          gs[2 * q + 1] = __fadd_rn(gs[2 * q + 1], pr[c][q].z);
          us[2 * q + 1] = __fadd_rn(us[2 * q + 1], pr[c][q].w);
        }
      }
#pragma unroll
      for (int e = 0; e < 8; e++) v[i][e] = on ? silu_mul_ieee(gs[e], us[e]) : 0.f;
    }
  }
  if (norm_w) {
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < KC; i++)
#pragma unroll
      for (int e = 0; e < 8; e++) ss += (double)v[i][e] * (double)v[i][e];
    ss = wave_sum_dpp_d(ss);
    __shared__ double red[kQuantThreads / 64];
    if ((t & 63) == 0) red[t >> 6] = ss;
    __syncthreads();
    ss = red[0] + red[1];
    const float inv = (float)(1.0 / sqrt(ss / K + (double)eps));
#pragma unroll
    for (int i = 0; i < KC; i++) {
      const int j = j0 + i * js;
      if (j < nch) {
        const float4 a = wpre[i][0], b = wpre[i][1];
        const float w8[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int e = 0; e < 8; e++) v[i][e] = w8[e] * (v[i][e] * inv);
      }
    }
  }
  if (xn_out && m >= M - xn_rows) {
    float4 *xo = reinterpret_cast<float4 *>(xn_out + (size_t)(m - (M - xn_rows)) * K);
#pragma unroll
    for (int i = 0; i < KC; i++) {
      const int j = j0 + i * js;
      if (j < nch) {
        xo[2 * j] = make_float4(v[i][0], v[i][1], v[i][2], v[i][3]);
        xo[2 * j + 1] = make_float4(v[i][4], v[i][5], v[i][6], v[i][7]);
      }
    }
  }
  if (!xq) return;
#pragma unroll
  for (int i = 0; i < KC; i++) {
    const int j = j0 + i * js;
    float amax = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[i][e]));
    // nch and the slice starts are multiples of 4, so a quad is wholly inside
    // or outside the row
    amax = quad_max_dpp(amax);
    if (j >= nch) continue;
    const float d = __fdiv_rn(amax, 127.0f);
    const float id = d != 0.f ? __fdiv_rn(1.0f, d) : 0.f;
    unsigned long long packed = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int q = (int)roundf(__fmul_rn(v[i][e], id));
      packed |= (unsigned long long)(uint8_t)(int8_t)q << (8 * e);
    }
    *reinterpret_cast<long *>(xq + qtile_offset(m, 8 * j, mt16)) = (long)packed;
    if ((j & 3) == 0) dx[qscale_offset(m, j >> 2, nb)] = (float)(_Float16)d;
  }
}

// The fused multiply-add chains over NB blocks from their operands, continuing
// acc: A av[i] (16 weight rows), B bv[t][i] (16 activation rows of tile t),
// the weight scales of the lane's 4 rows dwv[r][i] and the activation scales
// of its row dxv[t][i]: acc[t][r] = fma((float)dot, d_w * d_x, acc) in block
// order.
template <int TM, int NB>
__device__ __forceinline__ void chains(const long (&av)[NB], const long (&bv)[TM][NB],
                                       const float (&dwv)[4][NB], const float (&dxv)[TM][NB],
                                       float (&acc)[TM][4]) {
#pragma unroll
  for (int i = 0; i < NB; i++) {
#pragma unroll
    for (int t = 0; t < TM; t++) {
      const v4i ci =
          __builtin_amdgcn_mfma_i32_16x16x32_i8(av[i], bv[t][i], v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; r++)
        acc[t][r] = fmaf((float)ci[r], __fmul_rn(dwv[r][i], dxv[t][i]), acc[t][r]);
    }
  }
}

// The chains of NB blocks (b0 .. b0 + NB - 1, K % 512 == 0), continuing acc,
// for 16 weight rows from n0 and the activation tiles mt0 .. mt0 + TM - 1:
// acc[t][r] = output (n0 + 4 (lane / 16) + r, 16 (mt0 + t) + lane % 16); a
// tile past the last (mt16) repeats the last one and its outputs are not
// stored. All loads are unconditional and issued before the first MFMA (a
// guarded load would make the compiler wait for each one).
template <int TM, int NB>
__device__ __forceinline__ void chunk_chains(const int8_t *wq, const int8_t *xq, const float *dx,
                                             int N, int K, int n0, int mt0, int mt16, int b0,
                                             float (&acc)[TM][4]) {
  static_assert(NB % 8 == 0, "whole 8-block groups");
  constexpr int NH = NB / 8;  // 8-block groups of the weight scales
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int nb = K >> 5;
  const _Float16 *wd = reinterpret_cast<const _Float16 *>(wq + (size_t)N * K);
  const int4 *xq16 = reinterpret_cast<const int4 *>(xq);
  const int4 *wq16 = reinterpret_cast<const int4 *>(wq) + (size_t)(n0 >> 4) * K + lane;
  long av[NB], bv[TM][NB];
  float dwv[4][NB], dxv[TM][NB];
#pragma unroll
  for (int q = 0; q < NB / 2; q++) {  // blocks b0 + 2q, b0 + 2q + 1
    const int4 v = wq16[((b0 >> 1) + q) * 64];
    av[2 * q] = ((long)(unsigned)v.y << 32) | (unsigned)v.x;
    av[2 * q + 1] = ((long)(unsigned)v.w << 32) | (unsigned)v.z;
  }
#pragma unroll
  for (int t = 0; t < TM; t++) {
    const int tt = min(mt0 + t, mt16 - 1);
#pragma unroll
    for (int q = 0; q < NB / 2; q++) {
      const int4 v = xq16[((size_t)((b0 >> 1) + q) * mt16 + tt) * 64 + lane];
      bv[t][2 * q] = ((long)(unsigned)v.y << 32) | (unsigned)v.x;
      bv[t][2 * q + 1] = ((long)(unsigned)v.w << 32) | (unsigned)v.z;
    }
  }
#pragma unroll
  for (int r = 0; r < 4; r++)
#pragma unroll
    for (int h = 0; h < NH; h++) {
      const uint4 u =
          *reinterpret_cast<const uint4 *>(wd + (size_t)(n0 + 4 * g + r) * nb + b0 + 8 * h);
      const unsigned uw[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        dwv[r][8 * h + 2 * i] = (float)__builtin_bit_cast(_Float16, (unsigned short)(uw[i] & 0xffff));
        dwv[r][8 * h + 2 * i + 1] = (float)__builtin_bit_cast(_Float16, (unsigned short)(uw[i] >> 16));
      }
    }
#pragma unroll
  for (int t = 0; t < TM; t++) {
    const int tt = min(mt0 + t, mt16 - 1);
    const float4 *dp = reinterpret_cast<const float4 *>(dx + qscale_offset(tt * 16 + c, b0, nb));
#pragma unroll
    for (int q = 0; q < NB / 4; q++) {
      const float4 p = dp[16 * q];
      dxv[t][4 * q] = p.x, dxv[t][4 * q + 1] = p.y, dxv[t][4 * q + 2] = p.z, dxv[t][4 * q + 3] = p.w;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  chains<TM, NB>(av, bv, dwv, dxv, acc);
}

// y[m][n] (+)= sum_b d_w[n][b] d_x[m][b] sum_{k in b} q_w[n][k] q_x[m][k].
// A workgroup owns 16 weight rows (blockIdx.x) and TM 16-column activation
// tiles (blockIdx.y); its KW waves take the chunks in turn, each chunk's
// chains land in their own LDS slot, and the slots are added in chunk order.
// EPI_SWIGLU: rows 2j / 2j + 1 are gate / up of output j.
template <int TM, int KW, int EPI>
__global__ __launch_bounds__(KW * 64, 2) void k_gemm_i8(const int8_t *wq, const int8_t *xq,
                                                      float *y, int N, int K, int M, int ldy) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int nb = K >> 5, nch = nb / kChunkBlocks;
  const int mt16 = (M + 15) >> 4;
  const int n0 = blockIdx.x * 16, mt0 = blockIdx.y * TM;
  const float *dx = scales_of(const_cast<int8_t *>(xq), M, K);
  constexpr int LD = TM * 16 + 4;
  __shared__ float red[kMaxChunks][16][LD];
  for (int ch = w; ch < nch; ch += KW) {
    // a chunk's chain as two passes of 8 blocks (the second continues it):
    // TM tiles of 16 blocks would not fit the registers
    float acc[TM][4];
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[t][r] = 0.f;
    chunk_chains<TM, 8>(wq, xq, dx, N, K, n0, mt0, mt16, ch * kChunkBlocks, acc);
    chunk_chains<TM, 8>(wq, xq, dx, N, K, n0, mt0, mt16, ch * kChunkBlocks + 8, acc);
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) red[ch][4 * g + r][t * 16 + c] = acc[t][r];
  }
  __syncthreads();
  if (EPI == EPI_SWIGLU) {
    for (int idx = threadIdx.x; idx < TM * 16 * 8; idx += KW * 64) {
      const int ml = idx >> 3, p = idx & 7, m = mt0 * 16 + ml;
      float gs = 0.f, us = 0.f;
      for (int v = 0; v < nch; v++) {
        gs = __fadd_rn(gs, red[v][2 * p][ml]);
        us = __fadd_rn(us, red[v][2 * p + 1][ml]);
      }
      if (m < M) y[(size_t)m * ldy + (n0 >> 1) + p] = silu_mul_ieee(gs, us);
    }
  } else {
    for (int idx = threadIdx.x; idx < TM * 16 * 16; idx += KW * 64) {
      const int ml = idx >> 4, nl = idx & 15, m = mt0 * 16 + ml;
      float s = 0.f;
      for (int v = 0; v < nch; v++) s = __fadd_rn(s, red[v][nl][ml]);
      if (m < M) {
        float *yp = y + (size_t)m * ldy + n0 + nl;
        if (EPI == EPI_ADD)
          *yp = __fadd_rn(*yp, s);
        else
          *yp = s;
      }
    }
  }
}

// Many rows (a prompt's, or several prompts' together): a wave owns 64 weight
// rows x one activation tile and walks the whole K, the chain of each
// 512-column chunk in acc and the chunk sums added in chunk order in sum, so
// nothing meets in LDS. Per pair of 32-blocks the operands of both sides
// (coalesced 16-byte loads) are issued one pair ahead of the arithmetic, the
// activation scales two pairs ahead; the weight scales of a chunk go through
// the wave's own LDS as f32 (a lane needs those of four rows per block: one
// 16-byte read), loaded a chunk ahead. The four waves of a workgroup take
// consecutive weight rows of one activation tile (shared through the
// CU's L1). What bounds it is the scale chain: 12 VALU instructions (convert,
// multiply, fused multiply-add) per lane and MFMA, about three times the
// MFMA's own cycles.
template <int EPI>
__global__ __launch_bounds__(256, 2) void k_gemm_i8r(const int8_t *wq, const int8_t *xq, float *y,
                                                     int N, int K, int M, int ldy) {
  constexpr int NT = 4;
  __shared__ float dws[4][2][kChunkBlocks][16 * NT];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const int nb = K >> 5, np = K >> 6, nch = nb / kChunkBlocks, mt16 = (M + 15) >> 4;
  const int n0 = (blockIdx.x * 4 + wave) * 16 * NT, mt = blockIdx.y;
  const float *dx = scales_of(const_cast<int8_t *>(xq), M, K);
  const int4 *wt = reinterpret_cast<const int4 *>(wq) + (size_t)(n0 >> 4) * K + lane;
  // lane l loads (and writes to LDS) the scales of weight row n0 + l
  const uint4 *dwr = reinterpret_cast<const uint4 *>(
      reinterpret_cast<const _Float16 *>(wq + (size_t)N * K) + (size_t)(n0 + lane) * nb);
  const int4 *xt = reinterpret_cast<const int4 *>(xq) + (size_t)mt * 64 + lane;
  const float4 *dxr = reinterpret_cast<const float4 *>(dx + qscale_offset(16 * mt + c, 0, nb));
  int4 a[2][NT], b[2];
  float4 d4[2];
  uint4 dw[2];
  auto load = [&](int p, int s) {
    b[s] = xt[(size_t)p * mt16 * 64];
#pragma unroll
    for (int i = 0; i < NT; i++) a[s][i] = wt[(size_t)i * K + 64 * p];
  };
  auto load_dx = [&](int p, int s) { d4[s] = dxr[(p >> 1) * 16]; };  // blocks 2p .. 2p + 3, p even
  auto load_dw = [&](int ch) {
    dw[0] = dwr[2 * ch];
    dw[1] = dwr[2 * ch + 1];
  };
  auto store_dw = [&](int s) {
    const unsigned u[8] = {dw[0].x, dw[0].y, dw[0].z, dw[0].w, dw[1].x, dw[1].y, dw[1].z, dw[1].w};
#pragma unroll
    for (int i = 0; i < 8; i++) {
      dws[wave][s][2 * i][lane] = (float)__builtin_bit_cast(_Float16, (unsigned short)(u[i] & 0xffff));
      dws[wave][s][2 * i + 1][lane] = (float)__builtin_bit_cast(_Float16, (unsigned short)(u[i] >> 16));
    }
  };
  float acc[NT][4], sum[NT][4];
#pragma unroll
  for (int i = 0; i < NT; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) sum[i][r] = 0.f;
  load_dw(0);
  load(0, 0);
  load_dx(0, 0);
  store_dw(0);
  for (int ch = 0; ch < nch; ch++) {
    const int p0 = ch * (kChunkBlocks / 2);
    load_dw(min(ch + 1, nch - 1));
#pragma unroll
    for (int i = 0; i < NT; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[i][r] = 0.f;
    // the wave reads back only what it wrote itself (LDS keeps a wave's order)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < kChunkBlocks / 2; q++) {
      load(min(p0 + q + 1, np - 1), (q + 1) & 1);
      if ((q & 1) == 0) load_dx(min(p0 + q + 2, np - 2), ((q >> 1) + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; h++) {
        float4 dv[NT];
#pragma unroll
        for (int i = 0; i < NT; i++)
          dv[i] = *reinterpret_cast<const float4 *>(&dws[wave][ch & 1][2 * q + h][16 * i + 4 * g]);
        const float4 &dq = d4[(q >> 1) & 1];
        const float dxv = (q & 1) ? (h ? dq.w : dq.z) : (h ? dq.y : dq.x);
#pragma unroll
        for (int i = 0; i < NT; i++) {
          const v4i ci = __builtin_amdgcn_mfma_i32_16x16x32_i8(
              half_pair(a[q & 1][i], h), half_pair(b[q & 1], h), v4i{0, 0, 0, 0}, 0, 0, 0);
          const float dwv[4] = {dv[i].x, dv[i].y, dv[i].z, dv[i].w};
#pragma unroll
          for (int r = 0; r < 4; r++)
            acc[i][r] = fmaf((float)ci[r], __fmul_rn(dwv[r], dxv), acc[i][r]);
        }
      }
    }
    store_dw((ch + 1) & 1);
#pragma unroll
    for (int i = 0; i < NT; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) sum[i][r] = __fadd_rn(sum[i][r], acc[i][r]);
  }
  const int m = mt * 16 + c;
  if (m >= M) return;
#pragma unroll
  for (int i = 0; i < NT; i++) {
    const int n = n0 + 16 * i + 4 * g;
    const float(&s)[4] = sum[i];
    if (EPI == EPI_SWIGLU) {  // gate, up of outputs n / 2, n / 2 + 1
      *reinterpret_cast<float2 *>(y + (size_t)m * ldy + (n >> 1)) =
          make_float2(silu_mul_ieee(s[0], s[1]), silu_mul_ieee(s[2], s[3]));
    } else {
      float4 *yp = reinterpret_cast<float4 *>(y + (size_t)m * ldy + n);
      float4 v = make_float4(s[0], s[1], s[2], s[3]);
      if (EPI == EPI_ADD) {
        const float4 o = *yp;
        v = make_float4(__fadd_rn(o.x, s[0]), __fadd_rn(o.y, s[1]), __fadd_rn(o.z, s[2]),
                        __fadd_rn(o.w, s[3]));
      }
      *yp = v;
    }
  }
}

// One wave per (16 weight rows, chunk, TM activation tiles from TM z):
// part[chunk][m][n] = the chunk's chains. The waves of one (weight rows,
// chunk) over the row tiles are gridDim.x * gridDim.y workgroups apart (a
// multiple of 8 for the Qwen3-TTS shapes), so they run on one XCD and share
// the weight tile through its L2.
template <int TM>
__global__ __launch_bounds__(64, 2) void k_gemm_i8p(const int8_t *wq, const int8_t *xq,
                                                  float *part, int N, int K, int M) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int n0 = blockIdx.x * 16, ch = blockIdx.y, mt0 = blockIdx.z * TM;
  const int mt16 = (M + 15) >> 4;
  const float *dx = scales_of(const_cast<int8_t *>(xq), M, K);
  float acc[TM][4];
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) acc[t][r] = 0.f;
  chunk_chains<TM, kChunkBlocks>(wq, xq, dx, N, K, n0, mt0, mt16, ch * kChunkBlocks, acc);
#pragma unroll
  for (int t = 0; t < TM; t++) {
    const int m = (mt0 + t) * 16 + c;
    if (m < M)
      *reinterpret_cast<float4 *>(part + ((size_t)ch * M + m) * N + n0 + 4 * g) =
          make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
  }
}

// The gate/up product with SiLU(gate) * up and the quantization of the result
// fused: a workgroup owns 64 gate/up rows, i.e. one 32-block of the output,
// its 2 chunks (a wave per (16 rows, chunk), K == 1024) and the TM 16-row
// activation tiles from TM blockIdx.y; the chunk chains meet in LDS and are
// added in chunk order, then each row's block is quantized into yq (yq must
// not alias xq). The same values as k_gemm_i8p followed by
// k_quant_act<SRC_SWIGLU>. The workgroups of one output block over the row
// tiles are gridDim.x apart (a multiple of 8 for the Qwen3-TTS shapes: one
// XCD, one L2 for the weights).
template <int TM>
__global__ __launch_bounds__(512) void k_gemm_i8_swq(const int8_t *wq, const int8_t *xq,
                                                     int8_t *yq, int N, int M) {
  constexpr int K = 1024, LD = TM * 16 + 4, NCH = K / (32 * kChunkBlocks);
  __shared__ float red[NCH][64][LD];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int mt16 = (M + 15) >> 4, mt0 = blockIdx.y * TM;
  const int tile = w & 3, ch = w >> 2;  // 16-row tile of the 64, chunk
  const int n0 = blockIdx.x * 64 + tile * 16;
  const float *dx = scales_of(const_cast<int8_t *>(xq), M, K);
  float acc[TM][4];
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) acc[t][r] = 0.f;
  chunk_chains<TM, kChunkBlocks>(wq, xq, dx, N, K, n0, mt0, mt16, ch * kChunkBlocks, acc);
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) red[ch][tile * 16 + 4 * g + r][t * 16 + c] = acc[t][r];
  __syncthreads();
  // output block b = blockIdx.x of this workgroup's rows, 32 lanes per row
  const int KO = N >> 1, nbo = KO >> 5, b = blockIdx.x;
  float *dy = scales_of(yq, M, KO);
  const int nrow = min(TM, mt16 - mt0) * 16;
  for (int idx = threadIdx.x; idx < nrow * 32; idx += 64 * 4 * NCH) {
    const int ml = idx >> 5, j = idx & 31, m = mt0 * 16 + ml;
    float o = 0.f;
    if (m < M) {
      float gs = 0.f, us = 0.f;
#pragma unroll
      for (int v = 0; v < NCH; v++) {
        gs = __fadd_rn(gs, red[v][2 * j][ml]);
        us = __fadd_rn(us, red[v][2 * j + 1][ml]);
      }
      o = silu_mul_ieee(gs, us);
    }
    float amax = fabsf(o);
    amax = half_max_dpp(amax);
    const float d = __fdiv_rn(amax, 127.0f);
    const float id = d != 0.f ? __fdiv_rn(1.0f, d) : 0.f;
    yq[qtile_offset(m, 32 * b + j, mt16)] = (int8_t)(int)roundf(__fmul_rn(o, id));
    if (j == 0) dy[qscale_offset(m, b, nbo)] = (float)(_Float16)d;
  }
}

template <int TM, int KW>
void gemm_launch(const Mat &W, const QAct &xa, int M, int epi, float *y, int ldy,
                 hipStream_t st) {
  const int mt16 = (M + 15) >> 4;
  const dim3 grid(W.N / 16, (mt16 + TM - 1) / TM), block(KW * 64);
#define Q3H_GEMM(E)                                                                           \
  hipLaunchKernelGGL((k_gemm_i8<TM, KW, E>), grid, block, 0, st, W.q, xa.q, y, W.N, W.K, M, \
                     ldy)
  if (epi == EPI_STORE)
    Q3H_GEMM(EPI_STORE);
  else if (epi == EPI_ADD)
    Q3H_GEMM(EPI_ADD);
  else
    Q3H_GEMM(EPI_SWIGLU);
#undef Q3H_GEMM
}

template <int TM>
void gemm_by_k(const Mat &W, const QAct &xa, int M, int epi, float *y, int ldy, hipStream_t st) {
  // a wave per chunk
  const int nch = W.K / (32 * kChunkBlocks);
  if (nch >= 6)
    gemm_launch<TM, 6>(W, xa, M, epi, y, ldy, st);
  else if (nch >= 4)
    gemm_launch<TM, 4>(W, xa, M, epi, y, ldy, st);
  else
    gemm_launch<TM, 2>(W, xa, M, epi, y, ldy, st);
}

// Q8_0 quants [N][K] row-major to operand order (launch_tile_q8), 16 bytes (a
// lane's operands of a pair of blocks) per thread
__global__ __launch_bounds__(256) void k_tile_q8(const int8_t *__restrict__ src, int N, int K,
                                                 int8_t *__restrict__ dst) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)N * K / 16) return;
  const int lane = i & 63;
  const size_t tile = i >> 6;
  const int np = K >> 6, p = (int)(tile % np), n = (int)(tile / np) * 16 + (lane & 15);
  const int8_t *s = src + (size_t)n * K + 64 * p + 8 * (lane >> 4);
  const uint2 a = *reinterpret_cast<const uint2 *>(s), b = *reinterpret_cast<const uint2 *>(s + 32);
  reinterpret_cast<uint4 *>(dst)[i] = make_uint4(a.x, a.y, b.x, b.y);
}

void gemm_rows_launch(const Mat &W, const QAct &xa, int M, int epi, float *y, int ldy,
                      hipStream_t st) {
  const dim3 grid(W.N / 256, (M + 15) >> 4);
#define Q3H_GEMM(E)                                                                            \
  hipLaunchKernelGGL((k_gemm_i8r<E>), grid, dim3(256), 0, st, W.q, xa.q, y, W.N, W.K, M, ldy)
  if (epi == EPI_STORE)
    Q3H_GEMM(EPI_STORE);
  else if (epi == EPI_ADD)
    Q3H_GEMM(EPI_ADD);
  else
    Q3H_GEMM(EPI_SWIGLU);
#undef Q3H_GEMM
}

// slices > 1 only without a norm (each slice a whole number of 32-blocks)
template <int SRC, int NC>
void quant_launch_nc(float *x, const float *part, int ld, int M, int K, const float *norm_w,
                     float eps, const QAct &out, float *xn_out, int xn_rows, hipStream_t st,
                     int slices) {
  const int Mp = (M + 15) & ~15;
  const int kc = (K / 8 + kQuantThreads * slices - 1) / (kQuantThreads * slices);
  const dim3 grid(Mp, slices);
#define Q3H_QUANT(KC)                                                                          \
  hipLaunchKernelGGL((k_quant_act<SRC, KC, NC>), grid, dim3(kQuantThreads), 0, st, x, part,    \
                     out.q, norm_w, M, K, ld, eps, slices, xn_out, xn_rows)
  if (kc <= 1)
    Q3H_QUANT(1);
  else if (kc == 2)
    Q3H_QUANT(2);
  else
    Q3H_QUANT(3);
#undef Q3H_QUANT
}

template <int SRC>
void quant_launch(float *x, const float *part, int ld, int M, int K, const float *norm_w,
                  float eps, const QAct &out, float *xn_out, int xn_rows, hipStream_t st,
                  int slices = 1) {
  if (SRC == SRC_X || ld <= 2)
    quant_launch_nc<SRC, 2>(x, part, ld, M, K, norm_w, eps, out, xn_out, xn_rows, st, slices);
  else if (ld <= 4)
    quant_launch_nc<SRC, 4>(x, part, ld, M, K, norm_w, eps, out, xn_out, xn_rows, st, slices);
  else
    quant_launch_nc<SRC, 6>(x, part, ld, M, K, norm_w, eps, out, xn_out, xn_rows, st, slices);
}

}  // namespace

bool gemm_i8_supported(int N, int K) {
  return N > 0 && N % 16 == 0 && K > 0 && K % (32 * kChunkBlocks) == 0 &&
         K <= kQuantThreads * kQuantChunks * 8;
}

void launch_tile_q8(const int8_t *src, int N, int K, int8_t *dst, hipStream_t st) {
  const size_t n = (size_t)N * K / 16;
  hipLaunchKernelGGL(k_tile_q8, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, src, N, K,
                     dst);
}

int gemm_i8_chunks(int K) { return K / (32 * kChunkBlocks); }

size_t qact_bytes(int M, int K) {
  const size_t Mp = (M + 15) & ~15;
  return Mp * K + sizeof(float) * Mp * (K / 32);
}

void launch_quantize_act(const float *x, int ldx, int M, int K, const float *norm_w, float eps,
                         QAct out, float *xn_out, hipStream_t st, int xn_rows) {
  quant_launch<SRC_X>(const_cast<float *>(x), nullptr, ldx, M, K, norm_w, eps, out, xn_out,
                      xn_rows, st);
}

void launch_residual_quantize(float *h, const float *part, int chunks, int M, int K,
                              const float *norm_w, float eps, const QAct *out, hipStream_t st,
                              float *normed) {
  quant_launch<SRC_ADD>(h, part, chunks, M, K, norm_w, eps, out ? *out : QAct{}, normed, M, st);
}

void launch_swiglu_quantize(const float *part, int chunks, int M, int K, QAct out,
                            hipStream_t st) {
  const int slices = (K / 8 + kQuantThreads - 1) / kQuantThreads;
  quant_launch<SRC_SWIGLU>(nullptr, part, chunks, M, K, nullptr, 0.f, out, nullptr, 0, st,
                           slices);
}

// The waves of k_gemm_i8r are 64 weight rows x one activation tile over the
// whole K: taken from 768 of them (three quarters of the chip's SIMDs), with
// fewer the chunk-parallel k_gemm_i8 ends first. Measured, both after the
// operand-order weights: gate/up (96 waves a tile) 100 rows 8.5 / 7.5 us, 136
// rows 8.6 / 9.7; q/k/v (64) 136 rows 7.9 / 6.9, 203 rows 8.2 / 8.8; o_proj
// (16) 512 rows 13.6 / 11.1, 1024 rows 15.0 / 18.6, 4350 rows 48 / 68; gate/up
// at 4350 rows 126 / 170 us (275 before, 215 -> 435 TOPS). Two tiles a wave
// (weights loaded once for both) gave 120 there but 87 / 80 us on q/k/v.
// k_gemm_i8 takes one tile per workgroup up to 160 rows (70 rows: q/k/v 4.6
// against 5.3 us with two and 7.8 with four, 9.2 with row-major weights),
// two above (o_proj, 512 rows: 11.1 / 11.8).
void launch_gemm_i8(const Mat &W, const QAct &xa, int M, int epi, float *y, int ldy,
                    hipStream_t st) {
  const int mt16 = (M + 15) >> 4;
  if (W.N % 256 == 0 && (W.N / 64) * mt16 >= 768)
    gemm_rows_launch(W, xa, M, epi, y, ldy, st);
  else if (M <= 160)
    gemm_by_k<1>(W, xa, M, epi, y, ldy, st);
  else
    gemm_by_k<2>(W, xa, M, epi, y, ldy, st);
}

// Both products below take one 16-row activation tile per workgroup, the
// tiles on a grid dimension of their own: a tile's waves do the work of a
// 16-row product, and more rows add workgroups instead of lengthening each.
// Above 32 rows a wave takes two tiles (its weights loaded once for both):
// one tile per wave would put more workgroups than CUs on the gate/up product.
bool launch_gemm_i8_swiglu_quantize(const Mat &W, const QAct &xa, int M, QAct out,
                                    hipStream_t st) {
  if (M > 64 || W.K != 1024 || W.N % 64 != 0) return false;
  const int mt16 = (M + 15) >> 4;
  if (mt16 > 2)
    hipLaunchKernelGGL(k_gemm_i8_swq<2>, dim3(W.N / 64, (mt16 + 1) / 2), dim3(512), 0, st, W.q,
                       xa.q, out.q, W.N, M);
  else
    hipLaunchKernelGGL(k_gemm_i8_swq<1>, dim3(W.N / 64, mt16), dim3(512), 0, st, W.q, xa.q,
                       out.q, W.N, M);
  return true;
}

void launch_gemm_i8_partial(const Mat &W, const QAct &xa, int M, float *part, hipStream_t st) {
  const int mt16 = (M + 15) >> 4;
  if (mt16 > 2) {
    const dim3 grid(W.N / 16, gemm_i8_chunks(W.K), (mt16 + 1) / 2);
    hipLaunchKernelGGL(k_gemm_i8p<2>, grid, dim3(64), 0, st, W.q, xa.q, part, W.N, W.K, M);
  } else {
    const dim3 grid(W.N / 16, gemm_i8_chunks(W.K), mt16);
    hipLaunchKernelGGL(k_gemm_i8p<1>, grid, dim3(64), 0, st, W.q, xa.q, part, W.N, W.K, M);
  }
}

}  // namespace q3h
