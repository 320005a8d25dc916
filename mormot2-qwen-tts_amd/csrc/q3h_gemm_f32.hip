// q3h_gemm_f32.hip - the products of f32 stacks (the reference's f32 mode,
// lm.pas:177-178 with idtF32) over several rows, on the matrix cores:
// y[m][n] (+)= sum_k W[n][k] x[m][k], W row-major [N][K] f32, x [M][ldx].
//
// v_mfma_f32_16x16x4_f32 (wave64): lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16] of a 16x4 and a 4x16 operand and receives
// D[4 (l / 16) + r][l % 16], r < 4. Here A is 16 activation rows and B 16
// weight rows (as columns), both read straight from memory: lane l loads 16
// bytes, columns 4 (l / 16) .. + 3 of its row, of each 16-column step, so one
// load instruction covers 64 contiguous bytes of 16 rows, and the four floats
// feed four MFMAs (MFMA i takes column 4 (l / 16) + i of the step in k slot
// l / 16, the same for A and B, so the products pair up as in the sum).
// fp32 inputs, fp32 products and accumulation: no rounding of the operands.
//
// A workgroup owns 16 weight rows (n) and TM tiles of 16 activation rows (m);
// its K / 256 waves take 256 columns each, with the loads of up to 16
// 16-column steps in flight ahead of the MFMAs, and their partial sums meet in LDS
// in wave order (a fixed order: results do not depend on scheduling). The
// epilogue stores, adds to y (the residual), or applies SwiGLU to the
// interleaved gate / up rows (row 2j gate j, 2j + 1 up j: out[m][j] =
// silu(gate) * up). The grid covers all M rows in tiles of 16 TM, so a prefill
// of 512 rows is one launch per product; every tile reads the weights, which
// the later tiles find in L2 / Infinity Cache.
#include <hip/hip_runtime.h>

#include <climits>

#include "q3h_api_internal.h"
#include "q3h_math.h"
#include "q3h_wave.h"
#include "q3h_x3.h"

namespace q3h {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int KC = 256;  // columns per wave

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

__device__ __forceinline__ float silu_mul_f(float g, float u) { return g / (1.0f + expf(-g)) * u; }

typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));

// 8 Q8_0 quants (two dwords, little-endian bytes) as 8 bf16: the high halves
// of their f32 values, exact (at most 8 significant bits)
__device__ __forceinline__ bf8v q8_bf16x8(uint2 w) {
  const uint32_t w2[2] = {w.x, w.y};
  u32x4v o;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t word = w2[i >> 1], sh = 16 * (i & 1);
    const uint32_t f0 = __float_as_uint((float)(int8_t)(word >> sh));
    const uint32_t f1 = __float_as_uint((float)(int8_t)(word >> (sh + 8)));
    o[i] = (f0 >> 16) | (f1 & 0xffff0000u);
  }
  return __builtin_bit_cast(bf8v, o);
}

// the sums of a tile, met in LDS (red[wave][t][q][lane]: the MFMA result
// layout), added in wave order and stored / added / SwiGLU'd / kept as a slice
template <int TM, int KW, int EPI>
__device__ __forceinline__ void epilogue(const float (&red)[KW][TM][4][64], int m0, int n0, int M,
                                         float *__restrict__ y, int ldy) {
  // output (m, n) of this tile: t, lane' = 16 (m / 4 % 4) + n % 16, q = m % 4
  for (int o = threadIdx.x; o < TM * 256; o += 64 * KW) {
    const int t = o >> 8, q = (o >> 6) & 3, l = o & 63;
    const int m = m0 + 16 * t + 4 * (l >> 4) + q, n = n0 + (l & 15);
    if (m >= M) continue;
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < KW; i++) v += red[i][t][q][l];
    if (EPI == EPI_SWIGLU) {
      // gate in even rows, up in the odd row after it (the next lane)
      float u = 0.f;
#pragma unroll
      for (int i = 0; i < KW; i++) u += red[i][t][q][l ^ 1];
      if ((l & 1) == 0) y[(size_t)m * ldy + n / 2] = silu_mul_f(v, u);
    } else if (EPI == EPI_ADD) {
      y[(size_t)m * ldy + n] += v;
    } else if (EPI == EPI_ADD_SILU) {
      float *p = y + (size_t)m * ldy + n;
      *p = silu_clamp_f(*p + v);
    } else if (EPI == EPI_PART) {
      y[((size_t)blockIdx.z * M + m) * ldy + n] = v;
    } else {
      y[(size_t)m * ldy + n] = v;
    }
  }
}

// KK: the columns of one workgroup (K / gridDim.z; 256 per wave), K: the
// row stride of W. EPI_PART: the workgroup's sums go to slice blockIdx.z of
// y [gridDim.z][M][ldy] for a consumer that adds the slices in order.
template <int TM, int KK, int EPI>
__global__ __launch_bounds__(64 * (KK / KC)) void k_gemm_f32(const float *__restrict__ w,
                                                             const float *__restrict__ x,
                                                             int ldx, int M, int N, int K,
                                                             float *__restrict__ y, int ldy) {
  constexpr int KW = KK / KC;  // waves
  constexpr int ST = KC / 16;  // 16-column steps per wave
  __shared__ float red[KW][TM][4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (TM * 16);
  const int r = lane & 15, g = lane >> 4;
  const int kb = blockIdx.z * KK + wave * KC + 4 * g;
  const float *wr = w + (size_t)min(n0 + r, N - 1) * K + kb;
  const float *xr[TM];
#pragma unroll
  for (int t = 0; t < TM; t++) xr[t] = x + (size_t)min(m0 + 16 * t + r, M - 1) * ldx + kb;

  v4f acc[TM];
#pragma unroll
  for (int t = 0; t < TM; t++) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  // a ring of D steps in flight: the loads of step s + D are issued before
  // the MFMAs of step s (scheduling barriers keep the order, so each step
  // waits only for its own loads)
  constexpr int D = TM == 1 ? ST : (TM == 4 && KW > 8 ? 4 : 8);
  float4 wb[D], xb[D][TM];
#pragma unroll
  for (int s = 0; s < D; s++) {
    wb[s] = ld4(wr + 16 * s);
#pragma unroll
    for (int t = 0; t < TM; t++) xb[s][t] = ld4(xr[t] + 16 * s);
  }
#pragma unroll
  for (int s = 0; s < ST; s++) {
    const int c = s % D;
    const float4 wc = wb[c];
    float4 xc[TM];
#pragma unroll
    for (int t = 0; t < TM; t++) xc[t] = xb[c][t];
    if (s + D < ST) {
      wb[c] = ld4(wr + 16 * (s + D));
#pragma unroll
      for (int t = 0; t < TM; t++) xb[c][t] = ld4(xr[t] + 16 * (s + D));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < TM; t++) {
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xc[t].x, wc.x, acc[t], 0, 0, 0);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xc[t].y, wc.y, acc[t], 0, 0, 0);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xc[t].z, wc.z, acc[t], 0, 0, 0);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(xc[t].w, wc.w, acc[t], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int t = 0; t < TM; t++)
#pragma unroll
    for (int q = 0; q < 4; q++) red[wave][t][q][lane] = acc[t][q];
  __syncthreads();

  epilogue<TM, KW, EPI>(red, m0, n0, M, y, ldy);
}

// Many rows (prefill): a workgroup per 64 activation rows x 16 WN weight rows
// over the whole K, so that each activation chunk is read once per 16 WN
// weight rows instead of once per 16. Wave w owns weight rows n0 + 16 w ..
// + 15 and all 4 tiles of 16 activation rows. Per 32-column chunk: the
// activations (64 x 32) go through LDS (double buffered, one barrier per
// chunk), each wave's weights straight to registers; the loads of chunk c + 1
// are issued before the MFMAs of chunk c. Operands as in k_gemm_f32 (lane l:
// row l % 16, columns 4 (l / 16) .. + 3 of each 16-column step); the result
// tile of a wave is complete, so the epilogue needs no reduction.
//
// K-slices: workgroup z takes columns z kc .. z kc + kc - 1 (kc = K without a
// split); EPI_PART stores its sums to slice z of y [gridDim.z][M][ldy].
template <int WN, int EPI>
__global__ __launch_bounds__(64 * WN) void k_gemm_f32_m64(const float *__restrict__ w,
                                                          const float *__restrict__ x, int ldx,
                                                          int M, int N, int K, int kc,
                                                          float *__restrict__ y, int ldy) {
  constexpr int NT = 64 * WN, XS = 36;  // threads; LDS row stride (floats, padded)
  constexpr int XF4 = 64 * 32 / 4 / NT;  // float4 of an activation chunk per thread
  __shared__ float xs[2][64 * XS];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * WN + 16 * wave, m0 = blockIdx.y * 64;
  const int kz = blockIdx.z * kc;
  const float *wr = w + (size_t)min(n0 + r, N - 1) * K + kz + 4 * g;
  // activation chunk loads: float4 f = t + NT i of the 64 x 8 float4 chunk
  const float *xr[XF4];
  int xo[XF4];
#pragma unroll
  for (int i = 0; i < XF4; i++) {
    const int f = t + NT * i, row = f >> 3, c4 = f & 7;
    xr[i] = x + (size_t)min(m0 + row, M - 1) * ldx + kz + 4 * c4;
    xo[i] = row * XS + 4 * c4;
  }
  float4 xn[XF4], wn[2], wc[2];
  auto load = [&](int kc) {
#pragma unroll
    for (int i = 0; i < XF4; i++) xn[i] = ld4(xr[i] + kc);
    wn[0] = ld4(wr + kc);
    wn[1] = ld4(wr + kc + 16);
  };
  v4f acc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
  load(0);
#pragma unroll
  for (int i = 0; i < XF4; i++) *reinterpret_cast<float4 *>(&xs[0][xo[i]]) = xn[i];
  wc[0] = wn[0];
  wc[1] = wn[1];
  __syncthreads();
  const int nc = kc / 32;
  for (int c = 0; c < nc; c++) {
    const int b = c & 1;
    if (c + 1 < nc) load(32 * (c + 1));
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int tm = 0; tm < 4; tm++) {
        const float4 xa = *reinterpret_cast<const float4 *>(&xs[b][(16 * tm + r) * XS + 16 * s + 4 * g]);
        acc[tm] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa.x, wc[s].x, acc[tm], 0, 0, 0);
        acc[tm] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa.y, wc[s].y, acc[tm], 0, 0, 0);
        acc[tm] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa.z, wc[s].z, acc[tm], 0, 0, 0);
        acc[tm] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa.w, wc[s].w, acc[tm], 0, 0, 0);
      }
    }
    if (c + 1 < nc) {
#pragma unroll
      for (int i = 0; i < XF4; i++) *reinterpret_cast<float4 *>(&xs[b ^ 1][xo[i]]) = xn[i];
      wc[0] = wn[0];
      wc[1] = wn[1];
    }
    __syncthreads();
  }
  // lane l holds (m = m0 + 16 tm + 4 g + q, n = n0 + r)
  const int n = n0 + r;
#pragma unroll
  for (int tm = 0; tm < 4; tm++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int m = m0 + 16 * tm + 4 * g + q;
      const float v = acc[tm][q];
      if (EPI == EPI_SWIGLU) {
        const float u = __shfl_xor(v, 1);  // up: the odd row after its gate
        if (m < M && (r & 1) == 0) y[(size_t)m * ldy + n / 2] = silu_mul_f(v, u);
      } else if (m < M) {
        if (EPI == EPI_ADD)
          y[(size_t)m * ldy + n] += v;
        else if (EPI == EPI_ADD_SILU)
          y[(size_t)m * ldy + n] = silu_clamp_f(y[(size_t)m * ldy + n] + v);
        else if (EPI == EPI_PART)
          y[((size_t)blockIdx.z * M + m) * ldy + n] = v;
        else
          y[(size_t)m * ldy + n] = v;
      }
    }
}

// f32 weights [N][K] into x3 operand tiles, one thread per 8
__global__ __launch_bounds__(256) void k_split3(const float *__restrict__ f, int N, int K,
                                                uint16_t *__restrict__ x3) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < (size_t)N * K / 8) x3_tile_lane(f, N, K, i, x3);
}

// The same products with Q8_0 weights (int8 quants [N][K], then fp16 scales
// [N][K/32]) and f32 activations, on the bf16 matrix cores. A quant is an
// integer of at most 8 significant bits, exact in bf16; an activation is
// split exactly into three bf16 parts (split3). One 32-block of 16 weight
// rows and 16 activation rows is three v_mfma_f32_16x16x32_bf16 (low, middle,
// high part, each adding exact products in fp32) into a block sum, which is
// scaled by the weight row's fp16 block scale and added to the row's fp32
// sum: y = sum over blocks of d * (sum over the block of x q).
//
// Lane l holds, per block, the 8 quants 8 (l / 16) .. + 7 of weight row
// n0 + l % 16 (one 8-byte load) and the same 8 columns of activation row
// m0 + 16 t + l % 16 of each tile t (two 16-byte loads), and receives
// D[4 (l / 16) + q][l % 16]: the output layout of k_gemm_f32, whose
// epilogues this kernel shares. A workgroup owns 16 NB weight rows and TM
// tiles of 16 activation rows (the activations split once for the NB weight
// tiles); its waves take NBW blocks each. A wave issues the
// loads of all its weights and scales first, then of its activations D
// blocks ahead of the arithmetic, so that it waits for few memory round
// trips. (Its time is the activation loads: every workgroup reads all M rows
// over its K range; above 64 rows k_gemm_x3 shares them, already split.)
template <int KK>
constexpr int q8x_blocks_per_wave() {
  return KK <= 256 ? 2 : KK <= 1024 ? 4 : KK / 256;  // 4 to 8 waves
}

template <int TM, int KK, int EPI, int NB>
__global__ __launch_bounds__(64 * (KK / (32 * q8x_blocks_per_wave<KK>()))) void k_gemm_q8x(
    const int8_t *__restrict__ wq, const float *__restrict__ x, int ldx, int M, int N, int K,
    float *__restrict__ y, int ldy) {
  constexpr int NBW = q8x_blocks_per_wave<KK>();
  constexpr int KW = KK / (32 * NBW);     // waves
  constexpr int D = NBW < 4 ? NBW : 4;    // blocks in flight
  __shared__ float red[NB][KW][TM][4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = blockIdx.x * 16 * NB, m0 = blockIdx.y * (TM * 16);
  const int r = lane & 15, g = lane >> 4;
  const int kw = blockIdx.z * KK + wave * (32 * NBW);  // the wave's first column
  uint2 wv[NB][NBW];
  uint32_t dw[NB][NBW / 2];  // the block scales, 2 per dword
#pragma unroll
  for (int j = 0; j < NB; j++) {
    const int row = min(n0 + 16 * j + r, N - 1);
    const int8_t *wr = wq + (size_t)row * K + kw + 8 * g;
    const _Float16 *dr =
        reinterpret_cast<const _Float16 *>(wq + (size_t)N * K) + (size_t)row * (K / 32) + kw / 32;
#pragma unroll
    for (int b = 0; b < NBW; b++) wv[j][b] = *reinterpret_cast<const uint2 *>(wr + 32 * b);
    if constexpr (NBW == 2) {
      dw[j][0] = *reinterpret_cast<const uint32_t *>(dr);
    } else {
#pragma unroll
      for (int i = 0; i < NBW / 4; i++) {
        const uint2 t = *reinterpret_cast<const uint2 *>(dr + 4 * i);
        dw[j][2 * i] = t.x;
        dw[j][2 * i + 1] = t.y;
      }
    }
  }
  const float *xr[TM];
#pragma unroll
  for (int t = 0; t < TM; t++) xr[t] = x + (size_t)min(m0 + 16 * t + r, M - 1) * ldx + kw + 8 * g;

  u32x4v xb[D][TM][2];
  auto load = [&](int b, int c) {
#pragma unroll
    for (int t = 0; t < TM; t++) {
      xb[c][t][0] = *reinterpret_cast<const u32x4v *>(xr[t] + 32 * b);
      xb[c][t][1] = *reinterpret_cast<const u32x4v *>(xr[t] + 32 * b + 4);
    }
  };
#pragma unroll
  for (int s = 0; s < D; s++) load(s, s);
  v4f acc[NB][TM];
#pragma unroll
  for (int j = 0; j < NB; j++)
#pragma unroll
    for (int t = 0; t < TM; t++) acc[j][t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < NBW; b++) {
    const int c = b % D;
    u32x4v xc[TM][2];
#pragma unroll
    for (int t = 0; t < TM; t++) {
      xc[t][0] = xb[c][t][0];
      xc[t][1] = xb[c][t][1];
    }
    if (b + D < NBW) load(b + D, c);
    __builtin_amdgcn_sched_barrier(0);
    bf8v bw[NB];
    float d[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
      bw[j] = q8_bf16x8(wv[j][b]);
      d[j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(dw[j][b >> 1] >> (16 * (b & 1))));
    }
#pragma unroll
    for (int t = 0; t < TM; t++) {
      u32x4v ph, pm, pl;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const u32x4v &src = xc[t][i >> 1];
        uint32_t h0, m0_, l0, h1, m1, l1;
        split3(__uint_as_float(src[2 * (i & 1)]), h0, m0_, l0);
        split3(__uint_as_float(src[2 * (i & 1) + 1]), h1, m1, l1);
        ph[i] = h0 | (h1 << 16);
        pm[i] = m0_ | (m1 << 16);
        pl[i] = l0 | (l1 << 16);
      }
#pragma unroll
      for (int j = 0; j < NB; j++) {
        v4f s = v4f{0.f, 0.f, 0.f, 0.f};
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, pl), bw[j], s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, pm), bw[j], s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8v, ph), bw[j], s, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; q++) acc[j][t][q] = fmaf(d[j], s[q], acc[j][t][q]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int j = 0; j < NB; j++)
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
      for (int q = 0; q < 4; q++) red[j][wave][t][q][lane] = acc[j][t][q];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NB; j++) epilogue<TM, KW, EPI>(red[j], m0, n0 + 16 * j, M, y, ldy);
}

// Products over many rows (more than 64), the activations already split into
// operand tiles by the kernel that made them (x3_offset: RMSNorm, attention,
// SwiGLU), so that no product spends vector instructions on it: with the split
// in the staging of every 64 x 64 tile the Q8_0 products were bound by it (about
// 1200 VALU cycles to 384 of MFMA per 64 columns). Q8 == false: f32 weights in
// the same tiles (Mat::x3), six part products per chunk (x3 x x3, q3h_x3.h).
// Q8: int8 quants row-major and block scales; a quant is exact in bf16, so a
// 32-block is three part products into a block sum (low, middle, high part),
// scaled by the block scale into the fp32 sum.
//
// A workgroup of 4 waves owns 16 MT activation rows and 64 NT weight rows (NT
// 16-row tiles per wave) over the K range of its slice. Per step of KC 32-column
// chunks the activation tiles are copied to LDS (contiguous, two buffers, one
// barrier per step; loaded three steps ahead, through registers) and read as
// operands by every wave; the weights go to registers two steps ahead. A lane
// loads 16 quants of its row's 64 columns; v_permlane32_swap of the two halves
// leaves block 0 in the first and block 1 in the second, with the 8-column
// groups in the order 0, 2, 1, 3, which the activation operands are read in.
// The order of a row's sums is that of its chunks alone: any tile shape and
// row count gives the same bits.
template <bool Q8, int MT, int NT, int EPI>
struct GemmX3 {
  static constexpr int WN = 4, kThreads = 64 * WN, KC = Q8 ? 2 : 1;
  static constexpr int kStep = MT * KC * 192;           // 16-byte words of a step's activations
  static constexpr int kXW = (kStep + kThreads - 1) / kThreads;  // per thread
  static constexpr int kWW = Q8 ? 1 : 3;                // words per weight tile and step
  static constexpr int kOutLd = 8 * NT + 4;             // a wave's SwiGLU outputs in LDS
  static constexpr size_t kLds = 2 * kStep * 16;
  static_assert((size_t)WN * 16 * MT * kOutLd * 4 <= kLds, "the outputs fit the staging buffers");
};

template <bool Q8, int MT, int NT, int EPI>
__global__ __launch_bounds__(256, 2) void k_gemm_x3(const void *__restrict__ wp,
                                                    const uint16_t *__restrict__ x3, int M, int N,
                                                    int K, int kc, float *__restrict__ y, int ldy,
                                                    uint16_t *__restrict__ y3) {
  using G = GemmX3<Q8, MT, NT, EPI>;
  constexpr int KC = G::KC;
  __shared__ x3_u4 xs[2 * G::kStep];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = (blockIdx.x * G::WN + wave) * 16 * NT, mt0 = blockIdx.y * MT;
  const int nq = K >> 5, mt16 = (M + 15) >> 4;
  const int s0 = blockIdx.z * kc / (32 * KC), s1 = s0 + kc / (32 * KC);
  // this thread's words of a step: tile, then chunk, part and lane
  const x3_u4 *xg[G::kXW];
#pragma unroll
  for (int i = 0; i < G::kXW; i++) {
    const int f = min(t + G::kThreads * i, G::kStep - 1), tile = f / (KC * 192);
    xg[i] = reinterpret_cast<const x3_u4 *>(x3) + (size_t)min(mt0 + tile, mt16 - 1) * nq * 192 +
            (f - tile * KC * 192);
  }
  const int8_t *wq = reinterpret_cast<const int8_t *>(wp);
  const x3_u4 *wt = Q8 ? reinterpret_cast<const x3_u4 *>(wq + (size_t)(n0 + r) * K + 16 * g)
                       : reinterpret_cast<const x3_u4 *>(wp) + (size_t)(n0 >> 4) * nq * 192 + lane;
  const uint32_t *dr = reinterpret_cast<const uint32_t *>(
      reinterpret_cast<const _Float16 *>(wq + (size_t)N * K) + (size_t)(n0 + r) * nq);
  x3_u4 a[2][G::kXW], w[2][NT][G::kWW];
  uint32_t d[2][NT];
  auto load_x = [&](int s, int b) {
#pragma unroll
    for (int i = 0; i < G::kXW; i++) a[b][i] = xg[i][(size_t)min(s, s1 - 1) * KC * 192];
  };
  auto load_w = [&](int s, int b) {
    const int sc = min(s, s1 - 1);
#pragma unroll
    for (int j = 0; j < NT; j++) {
      if constexpr (Q8) {
        w[b][j][0] = wt[(size_t)j * K + 4 * sc];  // 16 rows of K bytes on: K words
        d[b][j] = dr[(size_t)j * 8 * nq + sc];
      } else {
#pragma unroll
        for (int c = 0; c < 3; c++) w[b][j][c] = wt[((size_t)j * nq + sc) * 192 + 64 * c];
      }
    }
  };
  auto stage = [&](int b, int sl) {
#pragma unroll
    for (int i = 0; i < G::kXW; i++) {
      const int f = t + G::kThreads * i;
      if (G::kStep % G::kThreads == 0 || f < G::kStep) xs[b * G::kStep + f] = a[sl][i];
    }
  };
  v4f acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; j++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[j][i] = v4f{0.f, 0.f, 0.f, 0.f};
  // f32 weights: the five products with a lower part have a sum of their own,
  // so that the sum of the high parts is rounded once per chunk and not six
  // times (error of a layer stack against float64: 1 layer, 71 rows 1.80e-7 ->
  // 1.56e-7, 1.76e-7 with f32 matrix cores in q/k/v and gate/up; 4 layers, 300
  // rows 3.9e-7 -> 2.9e-7; the same time)
  v4f low[Q8 ? 1 : NT][Q8 ? 1 : MT];
  if constexpr (!Q8) {
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < MT; i++) low[j][i] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  // the operand's lane in LDS: the 8-column groups in the weights' order
  const int la = Q8 ? ((g == 1 ? 2 : g == 2 ? 1 : g) * 16 + r) : lane;
  auto step = [&](int s, auto buf) {
    constexpr int b = decltype(buf)::value;
#pragma unroll
    for (int k = 0; k < KC; k++) {
      // (the operands of one chunk at a time: both took all 256 registers)
      if (KC > 1 && k) __builtin_amdgcn_sched_barrier(0);
      bf8v x[MT][3];
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int c = 0; c < 3; c++)
          x[i][c] = __builtin_bit_cast(bf8v, xs[b * G::kStep + ((i * KC + k) * 3 + c) * 64 + la]);
      if constexpr (Q8) {
#pragma unroll
        for (int j = 0; j < NT; j++) {
          const x3_u4 &q = w[b][j][0];
          const auto s0_ = __builtin_amdgcn_permlane32_swap(q[0], q[2], false, false);
          const auto s1_ = __builtin_amdgcn_permlane32_swap(q[1], q[3], false, false);
          const bf8v bw = q8_bf16x8(make_uint2(s0_[k], s1_[k]));
          const float dv = (float)__builtin_bit_cast(_Float16, (uint16_t)(d[b][j] >> (16 * k)));
          v4f sm[MT];
#pragma unroll
          for (int i = 0; i < MT; i++)
            sm[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[i][2], bw, v4f{0.f, 0.f, 0.f, 0.f},
                                                            0, 0, 0);
#pragma unroll
          for (int i = 0; i < MT; i++)
            sm[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[i][1], bw, sm[i], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < MT; i++)
            sm[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[i][0], bw, sm[i], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < MT; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[j][i][e] = fmaf(dv, sm[i][e], acc[j][i][e]);
        }
      } else {
        constexpr int pa[6] = {1, 2, 0, 1, 0, 0}, pb[6] = {1, 0, 2, 0, 1, 0};
#pragma unroll
        for (int c = 0; c < 6; c++)
#pragma unroll
          for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
              v4f &o = c < 5 ? low[j][i] : acc[j][i];
              o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  x[i][pa[c]], __builtin_bit_cast(bf8v, w[b][j][pb[c] % G::kWW]), o, 0, 0, 0);
            }
      }
    }
    load_w(s + 2, b);
    stage(b ^ 1, b ^ 1);
    load_x(s + 3, b ^ 1);
    __syncthreads();
  };
  load_x(s0, 0);
  load_w(s0, 0);
  load_x(s0 + 1, 1);
  load_w(s0 + 1, 1);
  stage(0, 0);
  load_x(s0 + 2, 0);
  __syncthreads();
  int s = s0;
  for (; s + 1 < s1; s += 2) {
    step(s, std::integral_constant<int, 0>{});
    step(s + 1, std::integral_constant<int, 1>{});
  }
  if (s < s1) step(s, std::integral_constant<int, 0>{});
  if constexpr (!Q8) {
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[j][i][e] += low[j][i][e];
  }
  // lane l holds (m = 16 (mt0 + i) + 4 g + e, n = n0 + 16 j + r)
  if constexpr (EPI == EPI_SWIGLU) {
    // silu(gate) * up through the wave's part of LDS (the steps are done: every
    // wave has passed the last barrier), then 8 columns per lane split into the
    // tiles of the next product's activations
    float *o = reinterpret_cast<float *>(xs) + wave * 16 * MT * G::kOutLd;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float v = acc[j][i][e], u = dpp_f<kQuadXor1>(v);
          if ((r & 1) == 0) o[(16 * i + 4 * g + e) * G::kOutLd + 8 * j + (r >> 1)] = silu_mul_f(v, u);
        }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int f = lane; f < 16 * MT * NT; f += 64) {
      const int row = f / NT, j = f % NT, m = 16 * mt0 + row;
      const float4 p0 = *reinterpret_cast<const float4 *>(&o[row * G::kOutLd + 8 * j]);
      const float4 p1 = *reinterpret_cast<const float4 *>(&o[row * G::kOutLd + 8 * j + 4]);
      const float v[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
      if (m < M) x3_store8(y3, m, n0 / 2 + 8 * j, N / 2, v, Q8);
    }
  } else {
    float *yo = y + (EPI == EPI_PART ? (size_t)blockIdx.z * M * ldy : 0) + n0 + r;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int m = 16 * (mt0 + i) + 4 * g + e;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < NT; j++) yo[(size_t)m * ldy + 16 * j] = acc[j][i][e];
      }
  }
}

// rows x [M][ldx] split into operand tiles, a thread per 4 columns
__global__ __launch_bounds__(256) void k_x3_rows(const float *__restrict__ x, int ldx, int M, int K,
                                                 uint16_t *__restrict__ o, bool cut) {
  const int i = blockIdx.x * 256 + threadIdx.x, m = i / (K / 4), k = 4 * (i - m * (K / 4));
  if (m >= M) return;
  const float4 v = ld4(x + (size_t)m * ldx + k);
  const float v4[4] = {v.x, v.y, v.z, v.w};
  x3_store4(o, m, k, K, v4, cut);
}

// h[m] += slices 0 .. S-1 of part [S][M][K], added in slice order (S == 0: h
// as it is); then, with a norm weight, w * (h[m] * inv), inv = 1 / sqrt(mean(
// h[m]^2) + eps) (sum of squares in double), to xn [M][K] or, split, to the
// operand tiles x3. One workgroup per row, K <= 4096, K % 4 == 0: a thread
// holds columns 4 t .. + 3 of each 1024-column round in registers (16-byte
// loads, all of a round issued together), and the norm weights are loaded
// before the partials, so the normalization needs no second trip to memory.
constexpr int kResidNormRounds = 4;

template <int S>
__global__ __launch_bounds__(256) void k_resid_norm(float *__restrict__ h,
                                                    const float *__restrict__ part, int M,
                                                    int K, const float *__restrict__ w,
                                                    float eps, float *__restrict__ xn,
                                                    uint16_t *__restrict__ x3, bool cut) {
  constexpr int NR = kResidNormRounds;
  __shared__ double red[4];
  // operand tiles: the 16 rows of a tile on one XCD (workgroups go to the XCDs
  // in turn), whose L2 joins their 16-byte pieces of each line
  const int b = blockIdx.x, t = threadIdx.x;
  const int m = x3 ? (b & ~127) + (b & 7) * 16 + ((b >> 3) & 15) : b;
  if (m >= M) return;
  float *hr = h + (size_t)m * K;
  float4 wv[NR], hv[NR];
  if (w) {
#pragma unroll
    for (int r = 0; r < NR; r++)
      if (1024 * r < K) wv[r] = ld4(w + min(1024 * r + 4 * t, K - 4));
  }
  double ss = 0.0;
#pragma unroll
  for (int r = 0; r < NR; r++) {
    if (1024 * r >= K) break;
    const int k = 1024 * r + 4 * t, kc = min(k, K - 4);
    float4 a[S ? S : 1];
#pragma unroll
    for (int s = 0; s < S; s++) a[s] = ld4(part + ((size_t)s * M + m) * K + kc);
    float4 v = ld4(hr + kc);
#pragma unroll
    for (int s = 0; s < S; s++) v.x += a[s].x, v.y += a[s].y, v.z += a[s].z, v.w += a[s].w;
    hv[r] = v;
    if (k < K) {
      if (S) *reinterpret_cast<float4 *>(hr + k) = v;
      ss += (double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z + (double)v.w * v.w;
    }
  }
  if (w == nullptr) return;
  for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off);
  if ((t & 63) == 0) red[t >> 6] = ss;
  __syncthreads();
  const double tot = red[0] + red[1] + red[2] + red[3];
  const float inv = (float)(1.0 / sqrt(tot / K + (double)eps));
#pragma unroll
  for (int r = 0; r < NR; r++) {
    const int k = 1024 * r + 4 * t;
    if (1024 * r >= K || k >= K) break;
    const float o[4] = {wv[r].x * (hv[r].x * inv), wv[r].y * (hv[r].y * inv),
                        wv[r].z * (hv[r].z * inv), wv[r].w * (hv[r].w * inv)};
    if (x3)
      x3_store4(x3, m, k, K, o, cut);
    else
      *reinterpret_cast<float4 *>(xn + (size_t)m * K + k) = make_float4(o[0], o[1], o[2], o[3]);
  }
}

template <int TM, int KK>
void launch_tk(const Mat &W, const float *x, int ldx, int M, int epi, float *y, int ldy, int ks,
               hipStream_t st) {
  const dim3 grid(W.N / 16, (M + 16 * TM - 1) / (16 * TM), ks), block(64 * (KK / KC));
#define Q3H_G(E)                                                                            \
  hipLaunchKernelGGL((k_gemm_f32<TM, KK, E>), grid, block, 0, st, W.f, x, ldx, M, W.N, W.K, \
                     y, ldy)
  if (epi == EPI_STORE)
    Q3H_G(EPI_STORE);
  else if (epi == EPI_ADD)
    Q3H_G(EPI_ADD);
  else if (epi == EPI_SWIGLU)
    Q3H_G(EPI_SWIGLU);
  else if (epi == EPI_PART)
    Q3H_G(EPI_PART);
  else if constexpr (KK >= 1024)
    Q3H_G(EPI_ADD_SILU);
  else
    require(false, Q3H_E_ARG, "EPI_ADD_SILU takes the whole K");
#undef Q3H_G
}

template <int TM>
void launch_t(const Mat &W, const float *x, int ldx, int M, int epi, float *y, int ldy, int ks,
              hipStream_t st) {
  switch (W.K / ks) {
    case 256: launch_tk<TM, 256>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    case 512: launch_tk<TM, 512>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    case 768: launch_tk<TM, 768>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    case 1024: launch_tk<TM, 1024>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    case 2048: launch_tk<TM, 2048>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    default: launch_tk<TM, 3072>(W, x, ldx, M, epi, y, ldy, ks, st); break;
  }
}

template <int WN>
void launch_m64(const Mat &W, const float *x, int ldx, int M, int epi, float *y, int ldy,
                hipStream_t st, int ks = 1) {
  const dim3 grid(W.N / (16 * WN), (M + 63) / 64, ks), block(64 * WN);
  const int kc = W.K / ks;
#define Q3H_G(E)                                                                               \
  hipLaunchKernelGGL((k_gemm_f32_m64<WN, E>), grid, block, 0, st, W.f, x, ldx, M, W.N, W.K, kc, \
                     y, ldy)
  if (epi == EPI_STORE)
    Q3H_G(EPI_STORE);
  else if (epi == EPI_ADD)
    Q3H_G(EPI_ADD);
  else if (epi == EPI_ADD_SILU)
    Q3H_G(EPI_ADD_SILU);
  else if (epi == EPI_PART)
    Q3H_G(EPI_PART);
  else
    Q3H_G(EPI_SWIGLU);
#undef Q3H_G
}

// Q8_0 weights: k_gemm_q8x over the whole K (KK = K: every epilogue but
// EPI_ADD_SILU) or over K slices of KK <= 1024 columns (EPI_PART)
template <int TM, int KK, int NB>
void launch_q8x_k(const Mat &W, const float *x, int ldx, int M, int epi, float *y, int ldy,
                  int ks, hipStream_t st) {
  const dim3 grid(W.N / (16 * NB), (M + 16 * TM - 1) / (16 * TM), ks),
      block(64 * (KK / (32 * q8x_blocks_per_wave<KK>())));
#define Q3H_Q(E)                                                                                 \
  hipLaunchKernelGGL((k_gemm_q8x<TM, KK, E, NB>), grid, block, 0, st, W.q, x, ldx, M, W.N, W.K, \
                     y, ldy)
  if (epi == EPI_PART) {
    if constexpr (KK <= 1024)
      Q3H_Q(EPI_PART);
    else
      require(false, Q3H_E_ARG, "Q8_0 K slices take at most 1024 columns");
  } else if constexpr (KK >= 1024) {
    if (epi == EPI_STORE)
      Q3H_Q(EPI_STORE);
    else if (epi == EPI_ADD)
      Q3H_Q(EPI_ADD);
    else if (epi == EPI_SWIGLU)
      Q3H_Q(EPI_SWIGLU);
    else
      require(false, Q3H_E_ARG, "EPI_ADD_SILU takes f32 weights");
  } else {
    require(false, Q3H_E_ARG, "Q8_0 products over a K slice store partial sums only");
  }
#undef Q3H_Q
}

// NB 16-row weight tiles per wave: two over more than 16 rows (each
// activation load then feeds twice the matrix-core work: 48-row prefill
// 1.92 -> 1.85 ms), one below (8 rows: 1.03 against 1.07 ms with two)
template <int TM, int NB>
void launch_q8x_t(const Mat &W, const float *x, int ldx, int M, int epi, float *y, int ldy,
                  int ks, hipStream_t st) {
  switch (W.K / ks) {
    case 256: launch_q8x_k<TM, 256, NB>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    case 512: launch_q8x_k<TM, 512, NB>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    case 768: launch_q8x_k<TM, 768, NB>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    case 1024: launch_q8x_k<TM, 1024, NB>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    case 2048: launch_q8x_k<TM, 2048, 1>(W, x, ldx, M, epi, y, ldy, ks, st); break;
    default: launch_q8x_k<TM, 3072, 1>(W, x, ldx, M, epi, y, ldy, ks, st); break;
  }
}

// The tile of a product over M rows, by rounds of 256 workgroups (one per CU)
// and the time of a round of each: 64 x 128 tiles 100, 64 x 64 58, 32 x 64 38
// (measured, K = 1024: f32 q/k/v at 2048 rows 4, 8 and 16 rounds 78, 88 and 114
// us; Q8_0 gate/up 6, 12 and 24 rounds 92, 111 and 142 us; 203 rows, f32 q/k/v:
// 1, 1 and 2 rounds 21.1, 14.8 and 14.3 us). 64 x 256 tiles spilled registers.
// Before (64 x 64 tiles that split their own activations), Q8_0: gate/up 172
// us at 2048 rows and 30.5 at 203; f32 q/k/v 34 us at 512 rows, 25 now.
template <bool Q8, int EPI>
void launch_x3(const Mat &W, const uint16_t *x3, int M, int ks, float *y, int ldy, uint16_t *y3,
               hipStream_t st) {
  const void *wp = Q8 ? (const void *)W.q : (const void *)W.x3;
  const int r32 = (M + 31) / 32, r64 = (M + 63) / 64, nb = W.N / 64;
  auto cost = [&](int tiles, int round) { return (tiles * ks + 255) / 256 * round; };
  const int c42 = nb % 2 == 0 ? cost(nb / 2 * r64, 100) : INT_MAX, c41 = cost(nb * r64, 58),
            c21 = cost(nb * r32, 38);
#define Q3H_X(MT, NT, R)                                                                        \
  hipLaunchKernelGGL((k_gemm_x3<Q8, MT, NT, EPI>), dim3(W.N / (64 * NT), R, ks), dim3(256), 0, \
                     st, wp, x3, M, W.N, W.K, W.K / ks, y, ldy, y3)
  if (c42 <= c41 && c42 <= c21)
    Q3H_X(4, 2, r64);
  else if (c41 < c21)
    Q3H_X(4, 1, r64);
  else
    Q3H_X(2, 1, r32);
#undef Q3H_X
}

// Q8_0 weights, f32 activations [M][ldx], over K slices of K / ks columns
void launch_q8x(const Mat &W, const float *x, int ldx, int M, int epi, float *y, int ldy, int ks,
                hipStream_t st) {
  if (M <= 16) {
    launch_q8x_t<1, 1>(W, x, ldx, M, epi, y, ldy, ks, st);
  } else if (W.N % 32 != 0) {
    if (M <= 32)
      launch_q8x_t<2, 1>(W, x, ldx, M, epi, y, ldy, ks, st);
    else
      launch_q8x_t<4, 1>(W, x, ldx, M, epi, y, ldy, ks, st);
  } else if (M <= 32) {
    launch_q8x_t<2, 2>(W, x, ldx, M, epi, y, ldy, ks, st);
  } else if (M <= 48) {
    launch_q8x_t<3, 2>(W, x, ldx, M, epi, y, ldy, ks, st);
  } else {
    launch_q8x_t<4, 2>(W, x, ldx, M, epi, y, ldy, ks, st);
  }
}

void launch_m(const Mat &W, const float *x, int ldx, int M, int epi, float *y, int ldy,
              hipStream_t st) {
  if (M > 32 && epi != EPI_PART && W.N % 64 == 0 && (W.N / 64) * ((M + 63) / 64) >= 256) {
    // many rows and wide products: 64-row tiles over the whole K (at least
    // 1024 waves; narrower products keep the K split over waves below, whose
    // waves each take a quarter to a twelfth of K)
    launch_m64<4>(W, x, ldx, M, epi, y, ldy, st);
    return;
  }
  if (M <= 16)
    launch_t<1>(W, x, ldx, M, epi, y, ldy, 1, st);
  else if (M <= 32)
    launch_t<2>(W, x, ldx, M, epi, y, ldy, 1, st);
  else
    launch_t<4>(W, x, ldx, M, epi, y, ldy, 1, st);
}

}  // namespace

void launch_split3(const Mat &m, hipStream_t st) {
  const size_t n = (size_t)m.N * m.K / 8;
  hipLaunchKernelGGL(k_split3, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, m.f, m.N, m.K,
                     m.x3);
}

bool gemm_x3_supported(const Mat &W, int ks) {
  return (W.q || W.x3) && W.N % 64 == 0 && W.K % (64 * ks) == 0;
}

void launch_gemm_x3(const Mat &W, const uint16_t *x3, int M, float *y, int ldy, hipStream_t st) {
  if (W.q)
    launch_x3<true, EPI_STORE>(W, x3, M, 1, y, ldy, nullptr, st);
  else
    launch_x3<false, EPI_STORE>(W, x3, M, 1, y, ldy, nullptr, st);
}

void launch_gemm_x3_swiglu(const Mat &W, const uint16_t *x3, int M, uint16_t *y3, hipStream_t st) {
  if (W.q)
    launch_x3<true, EPI_SWIGLU>(W, x3, M, 1, nullptr, 0, y3, st);
  else
    launch_x3<false, EPI_SWIGLU>(W, x3, M, 1, nullptr, 0, y3, st);
}

int launch_gemm_x3_part(const Mat &W, const uint16_t *x3, int M, float *part, hipStream_t st,
                        int ks) {
  if (W.q)
    launch_x3<true, EPI_PART>(W, x3, M, ks, part, W.N, nullptr, st);
  else
    launch_x3<false, EPI_PART>(W, x3, M, ks, part, W.N, nullptr, st);
  return ks;
}

void launch_x3_rows(const float *x, int ldx, int M, int K, uint16_t *o, bool cut,
                    hipStream_t st) {
  const size_t n = (size_t)M * (K / 4);
  hipLaunchKernelGGL(k_x3_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, ldx, M, K,
                     o, cut);
}

bool gemm_f32_supported(int N, int K) {
  return N % 16 == 0 && (K == 1024 || K == 2048 || K == 3072);
}

void launch_gemm_f32(const Mat &W, const float *x, int ldx, int M, int epi, float *y, int ldy,
                     hipStream_t st) {
  if (W.f)
    launch_m(W, x, ldx, M, epi, y, ldy, st);
  else
    launch_q8x(W, x, ldx, M, epi, y, ldy, 1, st);
}

bool gemm_f32_slices_supported(int N, int K) {
  const int kk = K / kF32Slices;
  return N % 16 == 0 && K % kF32Slices == 0 && (kk == 256 || kk == 512 || kk == 768 || kk == 1024);
}

int q8x_slices(const Mat &W, int M) {
  if (W.f || !W.q || M <= 16 || M > kQ8SliceRows || W.N % 32 != 0 || W.K % 256 != 0) return 0;
  const int ks = W.K / 256;  // a slice count launch_resid_norm takes
  return ks <= 4 || ks == 6 || ks == 8 || ks == 12 ? ks : 0;
}

int launch_gemm_f32_part(const Mat &W, const float *x, int ldx, int M, float *part,
                         hipStream_t st) {
  if (!W.f) {
    const int ks = q8x_slices(W, M) ? W.K / 256 : kF32Slices;
    launch_q8x(W, x, ldx, M, EPI_PART, part, W.N, ks, st);
    return ks;
  }
  if (M > 64 && W.N % 64 == 0)
    launch_m64<4>(W, x, ldx, M, EPI_PART, part, W.N, st, kF32Slices);
  else if (M <= 16)
    launch_t<1>(W, x, ldx, M, EPI_PART, part, W.N, kF32Slices, st);
  else if (M <= 32)
    launch_t<2>(W, x, ldx, M, EPI_PART, part, W.N, kF32Slices, st);
  else
    launch_t<4>(W, x, ldx, M, EPI_PART, part, W.N, kF32Slices, st);
  return kF32Slices;
}

void launch_resid_norm(float *h, const float *part, int M, int K, const float *norm_w,
                       float eps, float *xn, int slices, hipStream_t st, uint16_t *x3,
                       bool cut) {
  require(K <= 1024 * kResidNormRounds && K % 4 == 0, Q3H_E_ARG, "launch_resid_norm: K above 4096");
#define Q3H_RN(S)                                                                               \
  hipLaunchKernelGGL(k_resid_norm<S>, dim3(x3 ? (M + 127) / 128 * 128 : M), dim3(256), 0, st, h, \
                     part, M, K, norm_w, eps, xn, x3, cut)
  switch (slices) {
    case 0: Q3H_RN(0); break;
    case 1: Q3H_RN(1); break;
    case 2: Q3H_RN(2); break;
    case 3: Q3H_RN(3); break;
    case 4: Q3H_RN(4); break;
    case 6: Q3H_RN(6); break;
    case 8: Q3H_RN(8); break;
    case 12: Q3H_RN(12); break;
    default: require(false, Q3H_E_ARG, "launch_resid_norm: 0-4, 6, 8 or 12 slices");
  }
#undef Q3H_RN
}

}  // namespace q3h
