// q3h_x3.h - f32 x f32 products on the bf16 matrix cores: the operand tiles of
// the many-row products (k_gemm_x3, which walks them itself) and the walks of
// the decoder's convolutions (X3Walk, X3Short).
//
// Each operand is split into three bf16 parts, x = hi + mid + lo exactly, hi
// and mid rounded to nearest (split3_rn), and six part products are accumulated
// in fp32: hi hi in a sum of its own, and hi mid, mid hi, hi lo, lo hi, mid mid
// in another that is added to it at the end (of a slice). A bf16 product is
// exact in fp32; the three products left out weigh at most 2^-24 of the whole
// and cancel on average. The matrix cores cut off where they align a product
// with its sum, so with one sum every hi hi product of a chunk lost up to an
// fp32 unit downwards and met six roundings instead of one: a sample of seven
// one-term products of the decoder 1.5e-7 off (RMS, mean -1.2e-7), 7.1e-8 (mean
// 0) with two sums, 6.7e-8 on the f32 matrix cores; the decoder's samples 2.1e-6
// off float64 -> 8.9e-7 (2.3e-6 on the f32 matrix cores).
//
// v_mfma_f32_16x16x32_bf16: lane l holds A[l % 16][8 (l / 16) .. + 7] and
// B[8 (l / 16) .. + 7][l % 16] and receives D[4 (l / 16) + r][l % 16]. A is
// 16 activation rows, B 16 weight rows. The weights come pre-split in operand
// order (x3_offset): [16-row tile][32-column chunk][part][lane][8], so an
// operand is one coalesced 16-byte load per lane, straight to registers. The
// many-row products' activations come in the same tiles, written by the kernel
// that makes them (x3_store4 / x3_store8); the decoder's are split as they go to
// LDS, shared by the workgroup's waves.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "q3h_math.h"

namespace q3h {

typedef float x3_v4f __attribute__((ext_vector_type(4)));
typedef __bf16 x3_bf8 __attribute__((ext_vector_type(8)));
typedef unsigned int x3_u4 __attribute__((ext_vector_type(4)));

constexpr int kX3Stride = 40;  // LDS row of a unit, bf16 (32 + 8: 80 bytes)

// element (m, k) of part p (0 hi, 1 mid, 2 lo) of K-column rows in operand
// tiles; 8 columns from a multiple of 8 are 16 contiguous bytes
__host__ __device__ inline size_t x3_offset(int m, int k, int K) {
  return ((size_t)(m >> 4) * (K >> 5) + (k >> 5)) * 1536 + ((k & 31) >> 3) * 128 + (m & 15) * 8 +
         (k & 7);
}
constexpr int kX3Part = 512;  // elements from a part of a tile to the next

// An infinity among the N values of v: its parts become (+-1, 0, +-inf). The
// lowest part meets only the other operand's high part, whose sign is the
// operand's and which is 0 for 0 alone, so the product is the infinity (or the
// NaN) that the operands' product is; in the high part it would also meet the
// other's lower parts, which are 0 or of the other sign for ordinary values.
// h, m, l: the parts in pairs (split3_rn).
template <int N>
__device__ __forceinline__ void x3_infinite(const float (&v)[N], uint32_t (&h)[N / 2],
                                            uint32_t (&m)[N / 2], uint32_t (&l)[N / 2]) {
  float top = fabsf(v[0]);
#pragma unroll
  for (int e = 1; e < N; e++) top = fmaxf(top, fabsf(v[e]));
  if (__builtin_expect(top != __builtin_inff(), 1)) return;
#pragma unroll
  for (int e = 0; e < N; e++) {
    if (fabsf(v[e]) != __builtin_inff()) continue;
    const int sh = 16 * (e & 1);
    const uint32_t keep = ~(0xffffu << sh), sign = (__float_as_uint(v[e]) >> 31) << 15;
    h[e / 2] = (h[e / 2] & keep) | ((0x3f80u | sign) << sh);
    m[e / 2] &= keep;
    l[e / 2] = (l[e / 2] & keep) | ((0x7f80u | sign) << sh);
  }
}

// N values split, in pairs. cut: the parts cut off instead of rounded, for
// products with Q8_0 weights, which sum all three: there the chunk's sum is
// what the matrix cores cut off, and parts of one sign err less (4 layers, 203
// rows, 32 prompts: 2.31e-7 off float64, 2.36e-7 with rounded parts).
template <int N>
__device__ __forceinline__ void x3_split(const float (&v)[N], bool cut, uint32_t (&h)[N / 2],
                                         uint32_t (&m)[N / 2], uint32_t (&l)[N / 2]) {
#pragma unroll
  for (int e = 0; e < N / 2; e++) {
    if (cut) {
      uint32_t h1, m1, l1;
      split3(v[2 * e], h[e], m[e], l[e]);
      split3(v[2 * e + 1], h1, m1, l1);
      h[e] |= h1 << 16;
      m[e] |= m1 << 16;
      l[e] |= l1 << 16;
    } else {
      split3_rn(v[2 * e], v[2 * e + 1], h[e], m[e], l[e]);
    }
  }
  x3_infinite(v, h, m, l);
}

// 4 columns from k (a multiple of 4) of row m, split into the tiles at o
__device__ __forceinline__ void x3_store4(uint16_t *o, int m, int k, int K, const float (&v)[4],
                                          bool cut) {
  uint32_t h[2], md[2], l[2];
  x3_split(v, cut, h, md, l);
  uint16_t *d = o + x3_offset(m, k, K);
  *reinterpret_cast<uint2 *>(d) = make_uint2(h[0], h[1]);
  *reinterpret_cast<uint2 *>(d + kX3Part) = make_uint2(md[0], md[1]);
  *reinterpret_cast<uint2 *>(d + 2 * kX3Part) = make_uint2(l[0], l[1]);
}

// 8 columns from k (a multiple of 8)
__device__ __forceinline__ void x3_store8(uint16_t *o, int m, int k, int K, const float (&v)[8],
                                          bool cut) {
  uint32_t h[4], md[4], l[4];
  x3_split(v, cut, h, md, l);
  x3_u4 *d = reinterpret_cast<x3_u4 *>(o + x3_offset(m, k, K));
  d[0] = x3_u4{h[0], h[1], h[2], h[3]};
  d[kX3Part / 8] = x3_u4{md[0], md[1], md[2], md[3]};
  d[2 * kX3Part / 8] = x3_u4{l[0], l[1], l[2], l[3]};
}

// weights f [N][K] row-major into the operand tiles x3 (3 N K bf16; N % 16 ==
// 0, K % 32 == 0), or the same tiles unsplit (WF32): one thread per (tile,
// chunk, lane)
__device__ inline void x3_f32_lane(const float *f, int N, int K, size_t i, float *o) {
  const int lane = i & 63, nq = K >> 5;
  const size_t tq = i >> 6;
  const float *s = f + ((tq / nq) * 16 + (lane & 15)) * K + 32 * (tq % nq) + 8 * (lane >> 4);
  float *d = o + tq * 512 + lane * 4;
  for (int e = 0; e < 4; e++) {
    d[e] = s[e];
    d[256 + e] = s[4 + e];
  }
}

__device__ inline void x3_tile_lane(const float *f, int N, int K, size_t i, uint16_t *x3) {
  const int lane = i & 63, nq = K >> 5;
  const size_t tq = i >> 6;  // tile * nq + chunk
  const int q = (int)(tq % nq), n = (int)(tq / nq) * 16 + (lane & 15);
  const int k = 32 * q + 8 * (lane >> 4);
  const float *s = f + (size_t)n * K + k;
  const float v[8] = {s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7]};
  x3_store8(x3, n, k, K, v, false);
}

// The walk of WN waves over a product's columns: wave w owns NT 16-row weight
// tiles, all share MT 16-row activation tiles; acc[j][i]: the sums of weight
// tile j and activation tile i. The columns come in units of 32 channels of
// TAPS taps (a dilated convolution; TAPS = 1: a plain product), chunk u TAPS +
// k the channels of unit u at tap k, which reads the activation rows k dil
// further down. A unit's rows (16 MT + (TAPS - 1) dil of them, up to HALO more
// than the tile) are split and staged in LDS once for all its taps, in two
// buffers with one barrier per unit; the rows are loaded up to three units
// ahead of their use, the weights (registers) two chunks ahead. SUM: the units
// come in slices of su; each slice is summed alone in acc from zero and added
// to tot in order (what separate workgroups per slice and a reduction give).
// WF32: the weights as f32 in the same tile order, split in registers (2 / 3 of
// the bytes, for layers whose time is their weights' stream).
template <int MT, int NT, int WN, int TAPS, int HALO, bool WF32>
struct X3Walk {
  static constexpr int kThreads = 64 * WN;
  static constexpr int kRows = 16 * MT + HALO;
  static constexpr int kXF4 = (kRows * 8 + kThreads - 1) / kThreads;  // float4 per thread
  static constexpr int kPlane = kRows * kX3Stride;  // a part's plane in LDS
  static constexpr int kLds = 2 * 3 * kPlane;       // uint16_t
  static constexpr int kWords = WF32 ? 128 : 192;   // 16-byte words of a weight tile's chunk
  // units of rows in flight (eight tiles: one, their sums take the registers)
  static constexpr int kAhead = MT * NT >= 8 ? 1 : 2;

  // x: the tile's first row, channel 0 (row stride ld); rmax: its last row that
  // exists; t: the thread among the WN waves; u0 .. u1 - 1: the units; nu: the
  // barriers to take part in (units of the longest walk of the workgroup)
  template <bool SUM>
  static __device__ __forceinline__ void run(const float *__restrict__ x, int ld, int rmax, int dil,
                                             const x3_u4 *__restrict__ wt, size_t tile_stride,
                                             int t, int u0, int u1, int nu, int su, uint16_t *xs,
                                             x3_v4f (&acc)[NT][MT], x3_v4f (&tot)[NT][MT]) {
    const int lane = t & 63, r = lane & 15, g = lane >> 4;
    const int q1 = u1 * TAPS;
    int xo[kXF4];
#pragma unroll
    for (int i = 0; i < kXF4; i++) {
      const int f = t + kThreads * i;
      xo[i] = min(f >> 3, rmax) * ld + 4 * (f & 7);
    }
    float4 xr[kAhead][kXF4];
    x3_u4 w[2][NT][WF32 ? 2 : 3];
    x3_v4f low[NT][MT];  // the sums of the products with a lower part
    auto load_x = [&](int u, int s) {
      const float *p = x + 32 * min(u, u1 - 1);
#pragma unroll
      for (int i = 0; i < kXF4; i++) xr[s][i] = *reinterpret_cast<const float4 *>(p + xo[i]);
    };
    auto load_w = [&](int q, int s) {
      const x3_u4 *p = wt + (size_t)min(q, q1 - 1) * kWords;
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int k = 0; k < (WF32 ? 2 : 3); k++) w[s][j][k] = p[j * tile_stride + 64 * k];
    };
    auto stage = [&](int b, int s) {
#pragma unroll
      for (int i = 0; i < kXF4; i++) {
        const int f = t + kThreads * i;
        uint2 h, m, l;
        split3_rn(xr[s][i].x, xr[s][i].y, h.x, m.x, l.x);
        split3_rn(xr[s][i].z, xr[s][i].w, h.y, m.y, l.y);
        if (kRows * 8 % kThreads == 0 || f < kRows * 8) {
          uint16_t *d = xs + b * 3 * kPlane + (f >> 3) * kX3Stride + 4 * (f & 7);
          *reinterpret_cast<uint2 *>(d) = h;
          *reinterpret_cast<uint2 *>(d + kPlane) = m;
          *reinterpret_cast<uint2 *>(d + 2 * kPlane) = l;
        }
      }
    };
    auto unit = [&](int u, auto buf, auto par) {
      constexpr int b = decltype(buf)::value, p0 = decltype(par)::value;
#pragma unroll
      for (int k = 0; k < TAPS; k++) {
        constexpr int kParts = 3;
        const int wb = (p0 + k) & 1;
        x3_bf8 a[MT][kParts], bw[NT][kParts];
        const uint16_t *s = xs + b * 3 * kPlane + (r + k * dil) * kX3Stride + 8 * g;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
          for (int c = 0; c < kParts; c++)
            a[i][c] = __builtin_bit_cast(
                x3_bf8, *reinterpret_cast<const x3_u4 *>(s + c * kPlane + 16 * i * kX3Stride));
#pragma unroll
        for (int j = 0; j < NT; j++) {
          if constexpr (WF32) {
            x3_u4 part[3];
#pragma unroll
            for (int e = 0; e < 4; e++) {
              uint32_t h, m, l;
              split3_rn(__uint_as_float(w[wb][j][e >> 1][2 * (e & 1)]),
                        __uint_as_float(w[wb][j][e >> 1][2 * (e & 1) + 1]), h, m, l);
              part[0][e] = h;
              part[1][e] = m;
              part[2][e] = l;
            }
#pragma unroll
            for (int c = 0; c < kParts; c++) bw[j][c] = __builtin_bit_cast(x3_bf8, part[c]);
          } else {
#pragma unroll
            for (int c = 0; c < kParts; c++) bw[j][c] = __builtin_bit_cast(x3_bf8, w[wb][j][c]);
          }
        }
        // a part product of every tile before the next (independent sums back to
        // back), the small ones first
        constexpr int pa[6] = {1, 2, 0, 1, 0, 0}, pb[6] = {1, 0, 2, 0, 1, 0};
#pragma unroll
        for (int c = 0; c < 6; c++)
#pragma unroll
          for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
              x3_v4f &o = c < 5 ? low[j][i] : acc[j][i];
              o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][pa[c]], bw[j][pb[c]], o, 0, 0, 0);
            }
        load_w(u * TAPS + k + 2, wb);
      }
      if (SUM && (u + 1 - u0) % su == 0) {
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int i = 0; i < MT; i++) {
            acc[j][i] = acc[j][i] + low[j][i];
            tot[j][i] = u + 1 - u0 == su ? acc[j][i] : tot[j][i] + acc[j][i];
            acc[j][i] = low[j][i] = x3_v4f{0.f, 0.f, 0.f, 0.f};
          }
      }
    };
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < MT; i++) acc[j][i] = low[j][i] = x3_v4f{0.f, 0.f, 0.f, 0.f};
    constexpr int kOdd = kAhead - 1;  // slot of the odd units
    load_x(u0, 0);
    load_w(u0 * TAPS, 0);
    if (kOdd) load_x(u0 + 1, kOdd);
    load_w(u0 * TAPS + 1, 1);
    stage(0, 0);
    load_x(u0 + kAhead, 0);
    __syncthreads();
    // unit u: its products from buffer u & 1, unit u + 1 staged in the other
    for (int i = 0; i < nu; i += 2) {
      const int u = u0 + i;
      if (u < u1) unit(u, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
      stage(1, kOdd);
      load_x(u + 1 + kAhead, kOdd);
      __syncthreads();
      if (i + 1 >= nu) break;
      if (u + 1 < u1)
        unit(u + 1, std::integral_constant<int, 1>{}, std::integral_constant<int, TAPS & 1>{});
      stage(0, 0);
      load_x(u + 2 + kAhead, 0);
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < MT; i++) acc[j][i] = acc[j][i] + low[j][i];
    if (SUM) {
      const int n = u1 - u0, last = n % su;
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++)
          acc[j][i] = last == 0 ? tot[j][i] : (n < su ? acc[j][i] : tot[j][i] + acc[j][i]);
    }
  }
};

// The same sums for one slice of at most SU units, one 16-row activation tile
// and one 16-row weight tile per wave: the walk of calls of few rows, whose
// time is the latency of its loads. The rows of all units are loaded and staged
// at once, with one barrier, the first D chunks' weights in flight meanwhile.
template <int WN, int TAPS, int HALO, int SU, bool WF32>
struct X3Short {
  static constexpr int kThreads = 64 * WN;
  static constexpr int kRows = 16 + HALO;
  static constexpr int kUnitF4 = kRows * 8;
  static constexpr int kXF4 = (SU * kUnitF4 + kThreads - 1) / kThreads;
  static constexpr int kPlane = kRows * kX3Stride;
  static constexpr int kLds = SU * 3 * kPlane;  // uint16_t
  static constexpr int kWords = WF32 ? 128 : 192;
  static constexpr int NC = SU * TAPS;
  static constexpr int D = NC < (WF32 ? 6 : 4) ? NC : (WF32 ? 6 : 4);

  static __device__ __forceinline__ x3_v4f run(const float *__restrict__ x, int ld, int rmax,
                                               int dil, const x3_u4 *__restrict__ wt, int t,
                                               int u0, int u1, uint16_t *xs) {
    const int lane = t & 63, r = lane & 15, g = lane >> 4, q1 = u1 * TAPS;
    float4 xr[kXF4];
    x3_u4 w[D][WF32 ? 2 : 3];
    auto load_w = [&](int c) {
      const x3_u4 *p = wt + (size_t)min(u0 * TAPS + c, q1 - 1) * kWords;
#pragma unroll
      for (int k = 0; k < (WF32 ? 2 : 3); k++) w[c % D][k] = p[64 * k];
    };
#pragma unroll
    for (int i = 0; i < kXF4; i++) {
      const int f = t + kThreads * i, u = f / kUnitF4, e = f - u * kUnitF4;
      xr[i] = *reinterpret_cast<const float4 *>(x + (size_t)min(e >> 3, rmax) * ld +
                                                32 * min(u0 + u, u1 - 1) + 4 * (e & 7));
    }
#pragma unroll
    for (int c = 0; c < D; c++) load_w(c);
#pragma unroll
    for (int i = 0; i < kXF4; i++) {
      const int f = t + kThreads * i, u = f / kUnitF4, e = f - u * kUnitF4;
      uint2 h, m, l;
      split3_rn(xr[i].x, xr[i].y, h.x, m.x, l.x);
      split3_rn(xr[i].z, xr[i].w, h.y, m.y, l.y);
      if (SU * kUnitF4 % kThreads == 0 || f < SU * kUnitF4) {
        uint16_t *d = xs + u * 3 * kPlane + (e >> 3) * kX3Stride + 4 * (e & 7);
        *reinterpret_cast<uint2 *>(d) = h;
        *reinterpret_cast<uint2 *>(d + kPlane) = m;
        *reinterpret_cast<uint2 *>(d + 2 * kPlane) = l;
      }
    }
    __syncthreads();
    x3_v4f acc = x3_v4f{0.f, 0.f, 0.f, 0.f}, low = acc;
#pragma unroll
    for (int c = 0; c < NC; c++) {
      constexpr int pa[6] = {1, 2, 0, 1, 0, 0}, pb[6] = {1, 0, 2, 0, 1, 0};
      const int u = c / TAPS, k = c % TAPS;
      x3_bf8 a[3], bw[3];
#pragma unroll
      for (int e = 0; e < 3; e++)
        a[e] = __builtin_bit_cast(x3_bf8, *reinterpret_cast<const x3_u4 *>(
                                              xs + u * 3 * kPlane + e * kPlane +
                                              (r + k * dil) * kX3Stride + 8 * g));
      if constexpr (WF32) {
        x3_u4 part[3];
#pragma unroll
        for (int e = 0; e < 4; e++) {
          uint32_t h, m, l;
          split3_rn(__uint_as_float(w[c % D][e >> 1][2 * (e & 1)]),
                    __uint_as_float(w[c % D][e >> 1][2 * (e & 1) + 1]), h, m, l);
          part[0][e] = h;
          part[1][e] = m;
          part[2][e] = l;
        }
#pragma unroll
        for (int e = 0; e < 3; e++) bw[e] = __builtin_bit_cast(x3_bf8, part[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 3; e++) bw[e] = __builtin_bit_cast(x3_bf8, w[c % D][e]);
      }
      if (c + D < NC) load_w(c + D);
      x3_v4f n = low;
#pragma unroll
      for (int e = 0; e < 5; e++)
        n = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[pa[e]], bw[pb[e]], n, 0, 0, 0);
      const x3_v4f hi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], bw[0], acc, 0, 0, 0);
      low = u0 + u < u1 ? n : low;
      acc = u0 + u < u1 ? hi : acc;
    }
    return acc + low;
  }
};

}  // namespace q3h
