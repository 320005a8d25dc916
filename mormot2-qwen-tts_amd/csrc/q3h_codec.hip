// q3h_codec.hip - the back part of the Qwen3-TTS 12 Hz decoder on the device
// (TQwenCodec.Back, src/tts/mormot.ai.tts.qwen.codec.pas:1040-1083, the pass
// TQwenCodecVulkan records, codec.vulkan.pas:568-652): two upsampling stages
// (transposed convolution 2 / 2, ConvNeXt), the input convolution, four
// blocks (SnakeBeta, transposed convolution of rate 8 / 5 / 4 / 3, three
// residual units of dilations 1 / 3 / 9), SnakeBeta, the output convolution
// and the clamp: 1920 samples per frame, ~2.4 GMAC.
//
// Every convolution (transposed ones included, rewritten as causal
// convolutions of taps K / stride whose stride x out output columns are the
// stride output rows) is one matrix-core product over an implicit im2col:
// output row t reads input rows t + k dil, k < taps, of a sequence buffer that
// holds the `past` history rows of the previous call on top of the new rows
// (TQwenVkSeq, codec.vulkan.pas:33-40). The f32 operands are split exactly into
// bf16 parts (q3h_x3.h). The columns of a product are walked in units of 32
// channels x all taps, so a unit's rows are staged once for its taps, in slices
// of a few units that are summed alone and then in order: the order of every
// sum depends only on the layer, not on the rows of the call, so decoding 1 + 3
// frames or 4 at once gives the same samples (the reference's property,
// codec.vulkan.pas:12-13). Measured (156 frames in passes of 16; one frame per
// call): 14.3 ms and 698 us with f32 MFMAs, partial sums of every 16 chunks
// through memory and sinf epilogues, 9.3 ms and 398 us.
//
// The elementwise steps ride in the products' epilogues: bias, GELU (erf),
// the residual add, the ConvNeXt layer scale, and SnakeBeta of the output
// written as the input of the next convolution (at its history offset). The
// depthwise convolution + LayerNorm of ConvNeXt is one kernel per row; the
// output convolution (96 -> 1) + clamp one thread per sample. At the end of a
// pass one kernel moves every sequence's last rows to its history.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "q3h_api_internal.h"
#include "q3h_x3.h"

namespace q3h {
namespace {

constexpr int kLatent = 1024, kDecDim = 1536, kFrameSamples = 1920;
constexpr int kRates[4] = {8, 5, 4, 3};
constexpr int kDils[3] = {1, 3, 9};

enum ConvEpi { CE_BIAS = 0, CE_GELU = 1, CE_RES = 2, CE_SCALED_RES = 3 };

struct ConvArgs {
  const float *x;  // sequence buffer [past + T][cin] (history rows first)
  const void *w;   // operand tiles (x3, or f32) of [n][taps cin], column 32 (u taps + k) + c % 32
                   // for channel c of unit u = c / 32 at tap k
  const float *b;  // [n]
  float *y;        // [T][n] or null
  const float *r;  // residual [T][n] (CE_RES, CE_SCALED_RES)
  const float *g;  // layer scale [n] (CE_SCALED_RES)
  float *z;        // SnakeBeta of the output [T][n] or null
  const float *sa, *sib;  // e^alpha, 1 / (e^beta + 1e-9), indexed by column % sc
  float *part;            // slice sums [slices][T][n] when the walk is split over workgroups
  int sc;
};

__device__ __forceinline__ float gelu(float v) {
  return 0.5f * v * (1.0f + erff(v * 0.70710678118654752f));
}

// SnakeBeta of v: v + sin(v e^alpha)^2 / (e^beta + 1e-9)
__device__ __forceinline__ float snake(float v, float sa, float sib) {
  return fmaf(sib, sin_squared(__fmul_rn(v, sa)), v);
}

// One workgroup: output rows m0 .. m0 + 16 MT - 1, columns n0 .. n0 + 16 NT WN
// - 1 (NT 16-column tiles per wave), on the bf16 matrix cores with both
// operands split exactly (X3Walk). The units of a layer are summed in fixed
// slices of su units, each alone and then in slice order, by
//  - CM_WALK: one set of waves, slice after slice;
//  - CM_GROUP: a set of waves per slice, their sums met in LDS;
//  - CM_PART: a workgroup per slice (blockIdx.z), its sums to a.part for
//    k_conv_reduce.
// Every output's sum has the same order in any tile and mode.
enum ConvMode { CM_WALK = 0, CM_GROUP = 1, CM_PART = 2 };

// SU > 0: one slice of at most SU units over one 16-row tile (X3Short), any mode.
template <int MT, int NT, int WN, int SG, int TAPS, bool WF32, int MODE, int SU>
struct ConvWalk {
  static constexpr int kHalo = (TAPS - 1) * (TAPS == 7 ? 9 : 1);  // (the largest dilation)
  using Walk = X3Walk<MT, NT, WN, TAPS, kHalo, WF32>;
  using Short = X3Short<WN, TAPS, kHalo, SU ? SU : 1, WF32>;
  static_assert(SU == 0 || (MT == 1 && NT == 1), "short slices: one tile per wave");
  static constexpr int kLds = SU ? Short::kLds : Walk::kLds;
  static constexpr int kWords = Walk::kWords;
};

template <int MT, int NT, int WN, int SG, int TAPS, bool WF32, int MODE, int SU>
__global__ __launch_bounds__(64 * WN * SG, SG > 2 ? 4 : 2) void k_conv_x3(
    const float *__restrict__ x, const void *__restrict__ w, int cin, int dil, int T, int n, int su,
    int epi, ConvArgs a) {
  using W = ConvWalk<MT, NT, WN, SG, TAPS, WF32, MODE, SU>;
  constexpr int kGroup = 64 * WN;
  constexpr int kSum = MT * NT * WN * 256;  // floats of a group's sums
  extern __shared__ uint16_t xs[];          // [SG][W::kLds]; then the groups' sums
  const int grp = SG > 1 ? threadIdx.x / kGroup : 0, t = threadIdx.x - grp * kGroup;
  const int lane = t & 63, wave = t >> 6;
  const int n0 = (blockIdx.x * WN + wave) * 16 * NT, m0 = blockIdx.y * 16 * MT;
  const int U = cin / 32;
  const int sl = MODE == CM_PART ? blockIdx.z : grp;
  const int u0 = MODE == CM_WALK ? 0 : sl * su, u1 = MODE == CM_WALK ? U : min(U, u0 + su);
  const size_t ts = (size_t)U * TAPS * W::kWords;  // 16-byte words of a weight tile
  const x3_u4 *wt = reinterpret_cast<const x3_u4 *>(w) + (size_t)(n0 >> 4) * ts + lane;
  x3_v4f acc[NT][MT];
  const float *xt = x + (size_t)m0 * cin;
  const int rmax = T - 1 - m0 + (TAPS - 1) * dil;
  if constexpr (SU > 0) {
    acc[0][0] = W::Short::run(xt, cin, rmax, dil, wt, t, u0, u1, xs + grp * W::kLds);
    if (MODE == CM_GROUP) __syncthreads();
  } else {
    x3_v4f tot[NT][MT];
    W::Walk::template run<MODE == CM_WALK>(xt, cin, rmax, dil, wt, ts, t, u0, u1,
                                           MODE == CM_WALK ? U : su, su, xs + grp * W::kLds, acc,
                                           tot);
  }
  const int r = lane & 15, g = lane >> 4;
  if constexpr (MODE == CM_PART) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int m = m0 + 16 * i + 4 * g + q;
        if (m >= T) continue;
#pragma unroll
        for (int j = 0; j < NT; j++)
          a.part[((size_t)blockIdx.z * T + m) * n + n0 + 16 * j + r] = acc[j][i][q];
      }
    return;
  }
  if constexpr (MODE == CM_GROUP) {
    // (the walk ended with a barrier: the staged rows are read)
    x3_v4f *ps = reinterpret_cast<x3_v4f *>(xs);
    if (grp > 0)
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++)
          ps[(grp - 1) * (kSum / 4) + (j * MT + i) * kGroup + t] = acc[j][i];
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int s = 1; s < SG; s++)
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++)
          acc[j][i] = acc[j][i] + ps[(s - 1) * (kSum / 4) + (j * MT + i) * kGroup + t];
  }
  // the epilogue: the residuals of all outputs are loaded together, before
  // anything is stored (a load behind a store to memory that could be the same
  // waits for it: 16 us of an epilogue at one frame were such waits)
  float rs[MT][4][NT], bias[NT], sa[NT], sib[NT], gs[NT];
  const bool snk = a.z != nullptr;
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const int nc = n0 + 16 * j + r;
    bias[j] = a.b[nc];
    sa[j] = snk ? a.sa[nc % a.sc] : 0.f;
    sib[j] = snk ? a.sib[nc % a.sc] : 0.f;
    gs[j] = epi == CE_SCALED_RES ? a.g[nc] : 0.f;
  }
  if (epi >= CE_RES) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int j = 0; j < NT; j++)
          rs[i][q][j] = a.r[(size_t)min(m0 + 16 * i + 4 * g + q, T - 1) * n + n0 + 16 * j + r];
  }
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int m = m0 + 16 * i + 4 * g + q;
      float v[NT], z[NT];
#pragma unroll
      for (int j = 0; j < NT; j++) {
        v[j] = __fadd_rn(acc[j][i][q], bias[j]);
        // GELU and the layer scale: ConvNeXt's layers, which are never walked
        if (MODE != CM_WALK && epi == CE_GELU) v[j] = gelu(v[j]);
        if (MODE != CM_WALK && epi == CE_SCALED_RES) v[j] = fmaf(gs[j], v[j], rs[i][q][j]);
        if (epi == CE_RES) v[j] = __fadd_rn(rs[i][q][j], v[j]);
        z[j] = snk ? snake(v[j], sa[j], sib[j]) : 0.f;
      }
      if (m < T) {
        const size_t o = (size_t)m * n + n0 + r;
#pragma unroll
        for (int j = 0; j < NT; j++) {
          if (a.y) a.y[o + 16 * j] = v[j];
          if (snk) a.z[o + 16 * j] = z[j];
        }
      }
    }
}

// f32 weights [n][K] into operand tiles (split, or f32), one thread per 8
__global__ __launch_bounds__(256) void k_conv_tiles(const float *__restrict__ f, int n, int K,
                                                    void *__restrict__ o, bool f32) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)n * K / 8) return;
  if (f32)
    x3_f32_lane(f, n, K, i, static_cast<float *>(o));
  else
    x3_tile_lane(f, n, K, i, static_cast<uint16_t *>(o));
}

// The slices of a split product (up to 16 of them loaded together) added in
// slice order, then the epilogue: bias, GELU / residual / layer scale, the
// stores to y and (SnakeBeta of the value) to z.
// (The operands of the first loads are plain arguments, preloaded in SGPRs.)
__global__ __launch_bounds__(256) void k_conv_reduce(const float *__restrict__ part, int S,
                                                     int plane, int n, int epi,
                                                     const float *__restrict__ b,
                                                     const float *__restrict__ rp, ConvArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= plane) return;
  const int c = i % n;
  const float bias = b[c];
  const float res = epi >= CE_RES ? rp[i] : 0.f, g = epi == CE_SCALED_RES ? a.g[c] : 0.f;
  float sa = 0.f, sib = 0.f;
  if (a.z) {
    sa = a.sa[c % a.sc];
    sib = a.sib[c % a.sc];
  }
  float v = 0.f;
  for (int s0 = 0; s0 < S; s0 += 16) {
    float p[16];
#pragma unroll
    for (int s = 0; s < 16; s++) p[s] = part[(size_t)min(s0 + s, S - 1) * plane + i];
#pragma unroll
    for (int s = 0; s < 16; s++)
      if (s0 + s < S) v = s0 + s ? __fadd_rn(v, p[s]) : p[s];
  }
  v = __fadd_rn(v, bias);
  if (epi == CE_GELU) v = gelu(v);
  if (epi == CE_RES) v = __fadd_rn(res, v);
  if (epi == CE_SCALED_RES) v = fmaf(g, v, res);
  if (a.y) a.y[i] = v;
  if (a.z) a.z[i] = snake(v, sa, sib);
}

// ConvNeXt's causal depthwise convolution (kernel 7) and LayerNorm (eps 1e-6)
// of row t: x [6 + T][1024] (history first) -> h [T][1024]. One workgroup of
// 256 threads per row, 4 channels per thread.
__global__ __launch_bounds__(256) void k_dw_ln(const float *__restrict__ x,
                                               const float *__restrict__ dw,
                                               const float *__restrict__ db,
                                               const float *__restrict__ nw,
                                               const float *__restrict__ nb,
                                               float *__restrict__ h) {
  __shared__ float red[2][4];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float v[4];
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int c = tid + 256 * j;
    float acc = db[c];
#pragma unroll
    for (int k = 0; k < 7; k++) acc = fmaf(dw[c * 7 + k], x[(size_t)(t + k) * kLatent + c], acc);
    v[j] = acc;
    s += acc;
  }
  for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
  if (lane == 0) red[0][wave] = s;
  __syncthreads();
  const float mean = ((red[0][0] + red[0][1]) + (red[0][2] + red[0][3])) * (1.0f / kLatent);
  float q = 0.f;
#pragma unroll
  for (int j = 0; j < 4; j++) q = fmaf(v[j] - mean, v[j] - mean, q);
  for (int off = 32; off >= 1; off >>= 1) q += __shfl_xor(q, off, 64);
  if (lane == 0) red[1][wave] = q;
  __syncthreads();
  const float var = ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3])) * (1.0f / kLatent);
  const float inv = 1.0f / sqrtf(var + 1e-6f);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int c = tid + 256 * j;
    h[(size_t)t * kLatent + c] = fmaf((v[j] - mean) * inv, nw[c], nb[c]);
  }
}

// the output convolution (96 -> 1, kernel 7) and the clamp: x [6 + T][96].
// Four lanes per sample, lane j over channels 24 j .. 24 j + 23 of the 7
// rows, the four sums joined as (p0 + p1) + (p2 + p3).
__global__ __launch_bounds__(256) void k_conv_out(const float *__restrict__ x,
                                                  const float *__restrict__ w,
                                                  float b, int T, float *__restrict__ pcm) {
  const int t = blockIdx.x * 64 + (threadIdx.x >> 2), j = threadIdx.x & 3;
  const int tc = min(t, T - 1);
  float acc = 0.f;
#pragma unroll
  for (int k = 0; k < 7; k++) {
    const float *xr = x + (size_t)(tc + k) * 96 + 24 * j;
    const float *wk = w + k * 96 + 24 * j;
#pragma unroll
    for (int c = 0; c < 24; c += 4) {
      const float4 xv = *reinterpret_cast<const float4 *>(xr + c);
      const float4 wv = *reinterpret_cast<const float4 *>(wk + c);
      acc = fmaf(wv.x, xv.x, acc);
      acc = fmaf(wv.y, xv.y, acc);
      acc = fmaf(wv.z, xv.z, acc);
      acc = fmaf(wv.w, xv.w, acc);
    }
  }
  const float p1 = __shfl_xor(acc, 1, 64);
  const float s01 = (j & 1) ? p1 + acc : acc + p1;  // p0 + p1 (p2 + p3) in both lanes
  const float s23 = __shfl_xor(s01, 2, 64);
  const float v = ((j & 2) ? s23 + s01 : s01 + s23) + b;
  if (j == 0 && t < T) pcm[t] = fminf(1.0f, fmaxf(-1.0f, v));
}

// a sequence buffer whose last `past` rows become its history
struct HistEntry {
  float *buf;
  int past, cols, mult;  // rows of the pass = frames x mult
};

// Rows T .. T + past - 1 move to 0 .. past - 1, a thread per 4 columns of a
// sequence (blockIdx.x) walking the rows in order, 18 at a time (histories are
// 1, 6, 18 or 54 rows): a batch is loaded whole before it is stored, and later
// batches read rows below every row stored before them, so rows that are both
// source and target (T < past) need no second buffer.
__global__ __launch_bounds__(64) void k_save_hist(const HistEntry *__restrict__ e, int frames) {
  const HistEntry h = e[blockIdx.x];
  const int T = frames * h.mult, c = (blockIdx.y * 64 + threadIdx.x) * 4;
  if (c >= h.cols) return;
  float *dst = global_ptr(h.buf) + c;
  const float *src = dst + (size_t)T * h.cols;
  constexpr int B = 18;
  for (int d0 = 0; d0 < h.past; d0 += B) {
    x3_v4f v[B];
#pragma unroll
    for (int j = 0; j < B; j++)
      v[j] = *reinterpret_cast<const x3_v4f *>(src + (size_t)min(d0 + j, h.past - 1) * h.cols);
#pragma unroll
    for (int j = 0; j < B; j++)
      if (d0 + j < h.past) *reinterpret_cast<x3_v4f *>(dst + (size_t)(d0 + j) * h.cols) = v[j];
  }
}

}  // namespace
}  // namespace q3h

using namespace q3h;

namespace {

// a convolution as the product kernels take it
struct DConv {
  void *w = nullptr;  // operand tiles: split, or f32
  float *b = nullptr;
  bool f32 = false;
  int su = 1;  // units per slice
  int cin = 0, n = 0, taps = 1, dil = 1;
};

struct DSnake {
  float *a = nullptr, *ib = nullptr;
};

struct DNext {
  float *dw = nullptr, *db = nullptr, *nw = nullptr, *nb = nullptr, *gamma = nullptr;
  DConv pw1, pw2;
};

struct DRes {
  DSnake a1, a2;
  DConv c1, c2;
};

struct DBlock {
  DSnake act;
  DConv up;
  DRes res[3];
  int cin = 0, cout = 0, rate = 0;
};

}  // namespace

struct q3h_codec {
  q3h_device *dev = nullptr;
  int max_frames = 0;
  hipStream_t stream = nullptr;
  std::vector<void *> allocs;
  int64_t bytes = 0;
  float *staging = nullptr;  // the weights of one layer as they are uploaded
  size_t staging_floats = 0;
  DConv up[2];
  DNext next[2];
  DConv conv0;
  DBlock blocks[4];
  DSnake act_out;
  float *out_w = nullptr;  // [7][96]
  float out_b = 0.f;
  // sequences (history rows first) and work buffers
  float *x_in = nullptr, *s_nx[2] = {nullptr, nullptr}, *x_mid = nullptr, *hn = nullptr,
        *gbuf = nullptr, *s_c0 = nullptr, *s_up[4] = {}, *xres[4] = {}, *s_r1[4][3] = {},
        *s_c2 = nullptr, *s_out = nullptr, *pcm = nullptr;
  float *part = nullptr;  // K-slice sums of the split products
  HistEntry *hist = nullptr;
  std::vector<HistEntry> hist_host;
  // the kernels of a pass of F frames, captured once per F and replayed
  std::vector<hipGraphExec_t> exec;  // [max_frames + 1]
  std::mutex mu;
};

namespace {

template <class T>
T *calloc_dev(q3h_codec *c, size_t n) {
  T *p = (T *)dev_alloc(sizeof(T) * (n ? n : 1));
  c->allocs.push_back(p);
  c->bytes += (int64_t)(sizeof(T) * n);
  check_hip(hipMemset(p, 0, sizeof(T) * (n ? n : 1)), "codec init");
  return p;
}

float *upload_f(q3h_codec *c, const std::vector<float> &v) {
  float *p = calloc_dev<float>(c, v.size());
  check_hip(hipMemcpy(p, v.data(), sizeof(float) * v.size(), hipMemcpyHostToDevice), "codec upload");
  return p;
}

// column of channel ch at tap k in the walk's order
inline size_t walk_column(int ch, int k, int taps) {
  return (size_t)((ch >> 5) * taps + k) * 32 + (ch & 31);
}

// A weight matrix v [n][taps cin], columns in the walk's order, as operand
// tiles. Layers of 1 to 4 rows per frame (the front ones, most of the weights)
// keep them as f32: a pass streams their weights once for at most a few row
// tiles.
void upload_tiles(q3h_codec *c, DConv &d, const std::vector<float> &v, bool front) {
  const size_t bytes = (front ? 4 : 6) * v.size();
  d.f32 = front;
  d.w = dev_alloc(bytes);
  c->allocs.push_back(d.w);
  c->bytes += (int64_t)bytes;
  if (c->staging_floats < v.size()) {
    dev_free(c->staging);
    c->staging = nullptr;
    c->staging_floats = 0;
    c->staging = (float *)dev_alloc(sizeof(float) * v.size());
    c->staging_floats = v.size();
  }
  check_hip(hipMemcpyAsync(c->staging, v.data(), sizeof(float) * v.size(), hipMemcpyHostToDevice,
                           c->stream),
            "codec upload");
  hipLaunchKernelGGL(k_conv_tiles, dim3((unsigned)((v.size() / 8 + 255) / 256)), dim3(256), 0,
                     c->stream, c->staging, d.n, d.taps * d.cin, d.w, front);
  check_hip(hipGetLastError(), "codec weight tiles");
  check_hip(hipStreamSynchronize(c->stream), "codec weight tiles");
  // units per slice: 6 to 14 chunks (a fixed split per layer)
  const int U = d.cin / 32;
  d.su = d.taps == 7 ? (U <= 3 ? 1 : 2) : (d.taps == 2 || U % 8 != 0 ? 6 : 8);
}

const float *need(const float *p, const char *what) {
  require(p != nullptr, Q3H_E_ARG, std::string("q3h_codec_create: NULL ") + what);
  return p;
}

// torch Conv1d weight [out][in][k]
DConv make_conv(q3h_codec *c, const float *w, const float *b, int cin, int out, int k, int dil,
                const char *what, bool front = false) {
  need(w, what);
  need(b, what);
  std::vector<float> wp((size_t)out * k * cin), bp(b, b + out);
  for (int o = 0; o < out; o++)
    for (int ch = 0; ch < cin; ch++)
      for (int j = 0; j < k; j++)
        wp[(size_t)o * k * cin + walk_column(ch, j, k)] = w[((size_t)o * cin + ch) * k + j];
  DConv d;
  d.b = upload_f(c, bp);
  d.cin = cin;
  d.n = out;
  d.taps = k;
  d.dil = dil;
  upload_tiles(c, d, wp, front);
  return d;
}

// torch ConvTranspose1d weight [in][out][K], K = taps x stride, as a causal
// convolution of `taps` over [history ; x]: output column j out + o of row t
// (the sample t stride + j), tap k reading input row t - (taps - 1 - k)
DConv make_tconv(q3h_codec *c, const float *w, const float *b, int cin, int out, int K,
                 int stride, const char *what, bool front = false) {
  need(w, what);
  need(b, what);
  const int taps = K / stride, n = stride * out;
  std::vector<float> wp((size_t)n * taps * cin), bp(n);
  for (int j = 0; j < stride; j++)
    for (int o = 0; o < out; o++) {
      bp[(size_t)j * out + o] = b[o];
      for (int k = 0; k < taps; k++) {
        const int i = taps - 1 - k;
        for (int ch = 0; ch < cin; ch++)
          wp[((size_t)j * out + o) * taps * cin + walk_column(ch, k, taps)] =
              w[((size_t)ch * out + o) * K + j + i * stride];
      }
    }
  DConv d;
  d.b = upload_f(c, bp);
  d.cin = cin;
  d.n = n;
  d.taps = taps;
  d.dil = 1;
  upload_tiles(c, d, wp, front);
  return d;
}

DConv make_linear(q3h_codec *c, const float *w, const float *b, int cin, int out,
                  const char *what) {
  return make_conv(c, w, b, cin, out, 1, 1, what, true);
}

DSnake make_snake(q3h_codec *c, const float *alpha, const float *beta, int n, const char *what) {
  need(alpha, what);
  need(beta, what);
  std::vector<float> a(n), ib(n);
  for (int i = 0; i < n; i++) {
    a[i] = expf(alpha[i]);
    ib[i] = 1.0f / (expf(beta[i]) + 1e-9f);
  }
  DSnake s;
  s.a = upload_f(c, a);
  s.ib = upload_f(c, ib);
  return s;
}

float *copy_vec(q3h_codec *c, const float *p, int n, const char *what) {
  need(p, what);
  return upload_f(c, std::vector<float>(p, p + n));
}

// the slices of a layer's product (fixed per layer)
int slices(const DConv &d) { return (d.cin / 32 + d.su - 1) / d.su; }

constexpr int kWalkWorkgroups = 256, kShortWorkgroups = 640;

template <int MT, int NT, int WN, int SG, int TAPS, bool WF32, int MODE, int SU = 0>
void conv_launch(q3h_codec *c, const DConv &d, const ConvArgs &a, int T, int epi, int S) {
  using W = ConvWalk<MT, NT, WN, SG, TAPS, WF32, MODE, SU>;
  const dim3 grid(d.n / (16 * NT * WN), (T + 16 * MT - 1) / (16 * MT), MODE == CM_PART ? S : 1);
  const size_t lds = std::max(sizeof(uint16_t) * SG * W::kLds,
                              sizeof(float) * (SG - 1) * MT * NT * WN * 256);
  auto *k = &k_conv_x3<MT, NT, WN, SG, TAPS, WF32, MODE, SU>;
  if (lds > (64 << 10))
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
              "codec LDS");
  hipLaunchKernelGGL(k, grid, dim3(64 * WN * SG), lds, c->stream, a.x, a.w, d.cin, d.dil, T, d.n,
                     d.su, epi, a);
}

// The modes of a layer of TAPS taps over T rows, nb its 16 WN-column blocks:
// one 16-row tile per slice and workgroup while these are few (calls of a
// frame, the front layers), the 2 to 4 slices of a layer as sets of waves of
// one workgroup (no partial sums through memory, no second launch); else 64-
// or 32-row tiles walked whole where they fill the chip, a workgroup per slice
// otherwise.
// (The kernels are built for the decoder's layers only: the front layers, f32
// tiles, have 4 and 16 slices at one tap, 6 to 16 otherwise; the blocks' transposed
// convolutions of two taps have 4, 2 and 1, their dilated convolutions 12, 6, 3
// and 3, and their pointwise ones 3, 2, 1 and 1.)
template <int WN, int TAPS, bool WF32, int SU>
bool conv_short(q3h_codec *c, const DConv &d, const ConvArgs &a, int T, int epi, int S) {
  const int tiles = (T + 15) / 16 * (d.n / (16 * WN));
  if (d.su != SU || tiles * (S > 4 ? S : 1) > kShortWorkgroups) return false;
  if constexpr (!WF32 && ((TAPS == 2 && WN == 3) || (TAPS == 1 && SU == 6)))
    if (S == 1) {
      conv_launch<1, 1, WN, 1, TAPS, WF32, CM_WALK, SU>(c, d, a, T, epi, S);
      return true;
    }
  if constexpr (!WF32 && WN == 4 && (TAPS == 2 || (TAPS == 1 && SU == 6)))
    if (S == 2) {
      conv_launch<1, 1, WN, 2, TAPS, WF32, CM_GROUP, SU>(c, d, a, T, epi, S);
      return true;
    }
  if constexpr (!WF32 && (TAPS == 7 || (TAPS == 1 && SU == 8)))
    if (S == 3) {
      conv_launch<1, 1, WN, 3, TAPS, WF32, CM_GROUP, SU>(c, d, a, T, epi, S);
      return true;
    }
  if constexpr (WN == 4 && (WF32 ? TAPS == 1 : TAPS == 2))
    if (S == 4) {
      conv_launch<1, 1, WN, 4, TAPS, WF32, CM_GROUP, SU>(c, d, a, T, epi, S);
      return true;
    }
  if constexpr (WN == 4 && (WF32 || (TAPS == 7 && SU == 2)))
    if (S > 4) {
      conv_launch<1, 1, WN, 1, TAPS, WF32, CM_PART, SU>(c, d, a, T, epi, S);
      return true;
    }
  return false;
}

// The rule's lines, measured on the four dilated convolutions of a 16-frame
// pass (us; columns per wave x rows per workgroup): n = 768, 512 rows: split
// 16 x 64 29.7, 32 x 64 30.9; n = 384, 2560 rows: walked 16 x 32 35, 16 x 64
// 43, split 32 x 64 30 + 6 for the reduction; n = 192, 10240 rows: walked 16 x
// 64 32, 16 x 32 39, 32 x 64 45 (320 workgroups on 256 CUs); n = 96, 30720
// rows: 32 x 64 (all columns) 26, 16 x 64 33. (With f32 MFMAs and partial sums
// through memory: 47 + 8 each.)
template <int WN, int TAPS, bool WF32>
void conv_mode(q3h_codec *c, const DConv &d, const ConvArgs &a, int T, int epi) {
  const int S = slices(d), r32 = (T + 31) / 32, r64 = (T + 63) / 64;
  const int nb = d.n / (16 * WN);
  bool done = false;
  if constexpr (TAPS == 7)
    done = conv_short<WN, TAPS, WF32, WN == 4 ? 2 : 1>(c, d, a, T, epi, S);
  else if constexpr (TAPS == 2)
    done = conv_short<WN, TAPS, WF32, 6>(c, d, a, T, epi, S);
  else
    done = (WN == 4 && conv_short<WN, TAPS, WF32, 8>(c, d, a, T, epi, S)) ||
           (!WF32 && conv_short<WN, TAPS, false, 6>(c, d, a, T, epi, S));
  if (done) {
    if (S <= 4) return;
  } else {
    if constexpr (!WF32) {
      if constexpr (WN == 3 && TAPS != 2)
        if (nb == 2 && r64 >= kWalkWorkgroups) {  // the whole width in one workgroup
          conv_launch<4, 2, WN, 1, TAPS, WF32, CM_WALK>(c, d, a, T, epi, S);
          return;
        }
      if (r64 * nb >= 448) {
        conv_launch<4, 1, WN, 1, TAPS, WF32, CM_WALK>(c, d, a, T, epi, S);
        return;
      }
      if (TAPS != 7 || r32 * nb >= kWalkWorkgroups) {
        conv_launch<2, 1, WN, 1, TAPS, WF32, CM_WALK>(c, d, a, T, epi, S);
        return;
      }
    }
    if constexpr (WN == 4 && (WF32 || TAPS == 7))
      conv_launch<4, 1, WN, 1, TAPS, WF32, CM_PART>(c, d, a, T, epi, S);
    else  // a layer of another shape
      require(false, Q3H_E_ARG, "codec: layer shape");
  }
  const int plane = T * d.n;
  hipLaunchKernelGGL(k_conv_reduce, dim3((plane + 255) / 256), dim3(256), 0, c->stream, a.part, S,
                     plane, d.n, epi, a.b, a.r, a);
}

// y / z of a product over T output rows of sequence x
void conv(q3h_codec *c, const DConv &d, const float *x, int T, float *y, int epi,
          const float *r = nullptr, const float *g = nullptr, float *z = nullptr,
          const DSnake *sn = nullptr, int sc = 1) {
  ConvArgs a{};
  a.x = x;
  a.w = d.w;
  a.b = d.b;
  a.y = y;
  a.r = r;
  a.g = g;
  a.z = z;
  a.sa = sn ? sn->a : nullptr;
  a.sib = sn ? sn->ib : nullptr;
  a.sc = sc;
  a.part = c->part;
  require(d.n % 64 == 0 || (d.n % 48 == 0 && !d.f32), Q3H_E_ARG, "codec: layer width");
  const bool w4 = d.n % 64 == 0;
#define Q3H_C(TAPS)                                  \
  do {                                               \
    if (d.f32)                                       \
      conv_mode<4, TAPS, true>(c, d, a, T, epi);     \
    else if (w4)                                     \
      conv_mode<4, TAPS, false>(c, d, a, T, epi);    \
    else                                             \
      conv_mode<3, TAPS, false>(c, d, a, T, epi);    \
  } while (0)
  if (d.taps == 1)
    Q3H_C(1);
  else if (d.taps == 2)
    Q3H_C(2);
  else
    Q3H_C(7);
#undef Q3H_C
}

// one pass of F <= max_frames frames: x already in c->x_in, pcm to c->pcm
void pass(q3h_codec *c, int F) {
  hipStream_t st = c->stream;
  const int L = kLatent;
  // upsampling: transposed convolution 2 / 2 then ConvNeXt, twice
  const float *in = c->x_in;
  int rows = F;
  for (int i = 0; i < 2; i++) {
    float *seq = c->s_nx[i];  // 6 history rows, then 2 rows new rows
    conv(c, c->up[i], in, rows, seq + 6 * L, CE_BIAS);
    rows *= 2;
    hipLaunchKernelGGL(k_dw_ln, dim3(rows), dim3(256), 0, st, seq, c->next[i].dw, c->next[i].db,
                       c->next[i].nw, c->next[i].nb, c->hn);
    conv(c, c->next[i].pw1, c->hn, rows, c->gbuf, CE_GELU);
    float *out = i == 0 ? c->x_mid : c->s_c0 + 6 * L;
    conv(c, c->next[i].pw2, c->gbuf, rows, out, CE_SCALED_RES, seq + 6 * L, c->next[i].gamma);
    in = out;
  }
  // input convolution; its SnakeBeta (block 1's) written as block 1's input
  conv(c, c->conv0, c->s_c0, rows, nullptr, CE_BIAS, nullptr, nullptr,
       c->s_up[0] + kDecDim, &c->blocks[0].act, kDecDim);
  for (int b = 0; b < 4; b++) {
    DBlock &B = c->blocks[b];
    const int co = B.cout;
    // transposed convolution: the residual stream, and SnakeBeta of it as the
    // first unit's conv1 input
    conv(c, B.up, c->s_up[b], rows, c->xres[b], CE_BIAS, nullptr, nullptr,
         c->s_r1[b][0] + 6 * kDils[0] * co, &B.res[0].a1, co);
    rows *= B.rate;
    for (int u = 0; u < 3; u++) {
      DRes &R = B.res[u];
      // conv1 (dilated), SnakeBeta as conv2's input
      conv(c, R.c1, c->s_r1[b][u], rows, nullptr, CE_BIAS, nullptr, nullptr, c->s_c2, &R.a2, co);
      // conv2 + residual; SnakeBeta of the new stream for what comes next
      float *z;
      const DSnake *sn;
      if (u < 2) {
        z = c->s_r1[b][u + 1] + 6 * kDils[u + 1] * co;
        sn = &B.res[u + 1].a1;
      } else if (b < 3) {
        z = c->s_up[b + 1] + co;
        sn = &c->blocks[b + 1].act;
      } else {
        z = c->s_out + 6 * 96;
        sn = &c->act_out;
      }
      conv(c, R.c2, c->s_c2, rows, u < 2 ? c->xres[b] : nullptr, CE_RES, c->xres[b], nullptr, z,
           sn, co);
    }
  }
  hipLaunchKernelGGL(k_conv_out, dim3((rows + 63) / 64), dim3(256), 0, st, c->s_out, c->out_w,
                     c->out_b, rows, c->pcm);
  hipLaunchKernelGGL(k_save_hist, dim3((unsigned)c->hist_host.size(), kDecDim / 256), dim3(64), 0, st,
                     c->hist, F);
  check_hip(hipGetLastError(), "codec kernels");
}

// the pass of F frames as one graph launch (captured at its first use)
void run_pass(q3h_codec *c, int F) {
  hipGraphExec_t &e = c->exec[F];
  if (!e) {
    hipGraph_t g = capture_graph(c->stream, [&] { pass(c, F); });
    const hipError_t r = hipGraphInstantiate(&e, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    check_hip(r, "instantiate");
  }
  check_hip(hipGraphLaunch(e, c->stream), "graph launch");
}

void codec_release(q3h_codec *c) {
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (hipGraphExec_t e : c->exec)
    if (e) (void)hipGraphExecDestroy(e);
  for (void *p : c->allocs) dev_free(p);
  dev_free(c->staging);
  if (c->stream) (void)hipStreamDestroy(c->stream);
}

}  // namespace

extern "C" int q3h_codec_create(q3h_device *dev, const q3h_codec_weights *w, int max_frames,
                                q3h_codec **out) {
  q3h_codec *c = nullptr;
  const int rc = guard([&] {
    require(dev && w && out, Q3H_E_ARG, "q3h_codec_create: NULL argument");
    require(max_frames >= 1 && max_frames <= 64, Q3H_E_ARG,
            "q3h_codec_create: max_frames must be in 1..64");
    check_hip(hipSetDevice(dev->ordinal), "hipSetDevice");
    c = new q3h_codec();
    c->dev = dev;
    c->max_frames = max_frames;
    c->exec.assign(max_frames + 1, nullptr);
    check_hip(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking), "hipStreamCreate");
    const int L = kLatent;
    for (int i = 0; i < 2; i++) {
      c->up[i] = make_tconv(c, w->up_w[i], w->up_b[i], L, L, 2, 2, "upsample conv", true);
      DNext &n = c->next[i];
      n.dw = copy_vec(c, w->dw_w[i], 7 * L, "dwconv weight");
      n.db = copy_vec(c, w->dw_b[i], L, "dwconv bias");
      n.nw = copy_vec(c, w->norm_w[i], L, "norm weight");
      n.nb = copy_vec(c, w->norm_b[i], L, "norm bias");
      n.gamma = copy_vec(c, w->gamma[i], L, "gamma");
      n.pw1 = make_linear(c, w->pw1_w[i], w->pw1_b[i], L, 4 * L, "pwconv1");
      n.pw2 = make_linear(c, w->pw2_w[i], w->pw2_b[i], 4 * L, L, "pwconv2");
    }
    c->conv0 = make_conv(c, w->conv0_w, w->conv0_b, L, kDecDim, 7, 1, "decoder.0.conv",
                         true);
    for (int b = 0; b < 4; b++) {
      DBlock &B = c->blocks[b];
      const q3h_codec_block &bw = w->block[b];
      B.cin = kDecDim >> b;
      B.cout = kDecDim >> (b + 1);
      B.rate = kRates[b];
      B.act = make_snake(c, bw.act_alpha, bw.act_beta, B.cin, "block snake");
      B.up = make_tconv(c, bw.up_w, bw.up_b, B.cin, B.cout, 2 * B.rate, B.rate, "block conv",
                        b == 0);
      for (int u = 0; u < 3; u++) {
        const q3h_codec_res &rw = bw.res[u];
        B.res[u].a1 = make_snake(c, rw.a1_alpha, rw.a1_beta, B.cout, "act1");
        B.res[u].a2 = make_snake(c, rw.a2_alpha, rw.a2_beta, B.cout, "act2");
        B.res[u].c1 = make_conv(c, rw.c1_w, rw.c1_b, B.cout, B.cout, 7, kDils[u], "conv1");
        B.res[u].c2 = make_conv(c, rw.c2_w, rw.c2_b, B.cout, B.cout, 1, 1, "conv2");
      }
    }
    c->act_out = make_snake(c, w->out_alpha, w->out_beta, 96, "decoder.5");
    need(w->out_w, "decoder.6.conv weight");
    need(w->out_b, "decoder.6.conv bias");
    {
      std::vector<float> ow(7 * 96);
      for (int k = 0; k < 7; k++)
        for (int ch = 0; ch < 96; ch++) ow[k * 96 + ch] = w->out_w[ch * 7 + k];
      c->out_w = upload_f(c, ow);
      c->out_b = w->out_b[0];
    }
    dev_free(c->staging);
    c->staging = nullptr;
    c->staging_floats = 0;
    // sequences and work buffers for max_frames frames
    const size_t F = max_frames;
    c->x_in = calloc_dev<float>(c, F * L);
    c->s_nx[0] = calloc_dev<float>(c, (6 + 2 * F) * L);
    c->x_mid = calloc_dev<float>(c, 2 * F * L);
    c->s_nx[1] = calloc_dev<float>(c, (6 + 4 * F) * L);
    c->hn = calloc_dev<float>(c, 4 * F * L);
    c->gbuf = calloc_dev<float>(c, 4 * F * 4 * L);
    c->s_c0 = calloc_dev<float>(c, (6 + 4 * F) * L);
    std::vector<HistEntry> &h = c->hist_host;
    h.push_back({c->s_nx[0], 6, L, 2});
    h.push_back({c->s_nx[1], 6, L, 4});
    h.push_back({c->s_c0, 6, L, 4});
    size_t rin = 4, c2max = 0;
    for (int b = 0; b < 4; b++) {
      const DBlock &B = c->blocks[b];
      const size_t rout = rin * B.rate;
      c->s_up[b] = calloc_dev<float>(c, (1 + rin * F) * B.cin);
      h.push_back({c->s_up[b], 1, B.cin, (int)rin});
      c->xres[b] = calloc_dev<float>(c, rout * F * B.cout);
      for (int u = 0; u < 3; u++) {
        const int past = 6 * kDils[u];
        c->s_r1[b][u] = calloc_dev<float>(c, (past + rout * F) * B.cout);
        h.push_back({c->s_r1[b][u], past, B.cout, (int)rout});
      }
      c2max = std::max(c2max, rout * F * B.cout);
      rin = rout;
    }
    c->s_c2 = calloc_dev<float>(c, c2max);
    c->s_out = calloc_dev<float>(c, (6 + rin * F) * 96);
    h.push_back({c->s_out, 6, 96, (int)rin});
    c->pcm = calloc_dev<float>(c, rin * F);
    // the split products' slices: the largest S x T x n of any layer
    size_t pmax = 0;
    auto need_part = [&](const DConv &d, size_t T) {
      const int S = slices(d);
      if (S > 1) pmax = std::max(pmax, (size_t)S * T * d.n);
    };
    for (int i = 0; i < 2; i++) {
      need_part(c->up[i], (i + 1) * F);
      need_part(c->next[i].pw1, 2 * (i + 1) * F);
      need_part(c->next[i].pw2, 2 * (i + 1) * F);
    }
    need_part(c->conv0, 4 * F);
    size_t rr = 4;
    for (int b = 0; b < 4; b++) {
      need_part(c->blocks[b].up, rr * F);
      rr *= c->blocks[b].rate;
      for (int u = 0; u < 3; u++) {
        need_part(c->blocks[b].res[u].c1, rr * F);
        need_part(c->blocks[b].res[u].c2, rr * F);
      }
    }
    c->part = calloc_dev<float>(c, pmax);
    c->hist = calloc_dev<HistEntry>(c, h.size());
    check_hip(hipMemcpy(c->hist, h.data(), sizeof(HistEntry) * h.size(), hipMemcpyHostToDevice),
              "codec init");
    dev->bytes += c->bytes;
    dev->stacks++;
    *out = c;
  });
  if (rc != 0 && c) {
    codec_release(c);
    delete c;
  }
  return rc;
}

extern "C" int q3h_codec_reset(q3h_codec *c) {
  return guard([&] {
    require(c != nullptr, Q3H_E_ARG, "q3h_codec_reset: NULL codec");
    std::lock_guard<std::mutex> lk(c->mu);
    check_hip(hipSetDevice(c->dev->ordinal), "hipSetDevice");
    for (const HistEntry &h : c->hist_host)
      check_hip(hipMemsetAsync(h.buf, 0, sizeof(float) * h.past * h.cols, c->stream), "reset");
    check_hip(hipStreamSynchronize(c->stream), "reset sync");
  });
}

extern "C" int q3h_codec_back(q3h_codec *c, const float *x, int frames, float *pcm) {
  return guard([&] {
    require(c != nullptr, Q3H_E_ARG, "q3h_codec_back: NULL codec");
    require(frames >= 0, Q3H_E_ARG, "q3h_codec_back: negative frame count");
    if (frames == 0) return;
    require(x != nullptr && pcm != nullptr, Q3H_E_ARG, "q3h_codec_back: NULL x or pcm");
    std::lock_guard<std::mutex> lk(c->mu);
    check_hip(hipSetDevice(c->dev->ordinal), "hipSetDevice");
    for (int f0 = 0; f0 < frames; f0 += c->max_frames) {
      const int F = std::min(c->max_frames, frames - f0);
      check_hip(hipMemcpyAsync(c->x_in, x + (size_t)f0 * kLatent, sizeof(float) * F * kLatent,
                               hipMemcpyHostToDevice, c->stream),
                "upload x");
      run_pass(c, F);
      check_hip(hipMemcpyAsync(pcm + (size_t)f0 * kFrameSamples, c->pcm,
                               sizeof(float) * F * kFrameSamples, hipMemcpyDeviceToHost, c->stream),
                "download pcm");
    }
    check_hip(hipStreamSynchronize(c->stream), "codec sync");
  });
}

extern "C" int64_t q3h_codec_bytes(const q3h_codec *c) { return c ? c->bytes : 0; }

extern "C" int q3h_codec_destroy(q3h_codec *c) {
  return guard([&] {
    if (!c) return;
    check_hip(hipSetDevice(c->dev->ordinal), "hipSetDevice");
    c->dev->bytes -= c->bytes;
    c->dev->stacks--;
    codec_release(c);
    delete c;
  });
}
