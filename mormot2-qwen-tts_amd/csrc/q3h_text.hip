// q3h_text.hip - the talker's text projection on the device
// (TQwenTalker.TextProject, src/tts/mormot.ai.tts.qwen.talker.pas:390-421):
// y[r] = fc2 . SiLU(fc1 . emb[ids[r]] + b1) + b2, SiLU(v) = 0 below -80.
//
// Five launches over all n rows at once: the rows of the embedding (BF16 is the
// high half of an f32: exact) split into operand tiles (k_text_rows); fc1 on
// the bf16 matrix cores with both operands split exactly (k_gemm_x3), K in 8
// slices so that its workgroups fill the chip at the row counts of a prompt;
// the slices added to b1, SiLU, split for fc2 (k_text_mid); fc2; the slices
// added to b2 (k_text_end). The products are as exact as fp32 ones (q3h_x3.h;
// the reference's idtF32 products): a result of two one-term products 3.6e-8 off
// float64 (RMS) as on the f32 matrix cores. 48 rows: 48 us of kernels as
// three launches on the f32 matrix cores, whose 128 and 64 workgroups walked
// all of K (23 + 20 us); widths that are no multiples of 64 and 512 still take
// those: e = the rows, h = b1, y = b2, then fc1 with h = SiLU(h + sum)
// (EPI_ADD_SILU) and fc2 with y += sum (EPI_ADD). The embedding table stays in the dtype it came in (BF16: 622 MB for 151936 x
// 2048), gathered one row per token.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>

#include "q3h_api_internal.h"
#include "q3h_math.h"
#include "q3h_x3.h"

namespace q3h {
namespace {

__device__ __forceinline__ float bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// one workgroup per row: e[r] = emb[ids[r]] in f32, h[r] = b1, y[r] = b2
// (TH % 8 == 0, H % 4 == 0; rows 16-byte aligned)
template <bool BF16>
__global__ __launch_bounds__(256) void k_text_rows(const void *__restrict__ emb,
                                                   const int32_t *__restrict__ ids, int TH,
                                                   int H, const float *__restrict__ b1,
                                                   const float *__restrict__ b2,
                                                   float *__restrict__ e, float *__restrict__ h,
                                                   float *__restrict__ y, int ldy) {
  const int r = blockIdx.x, t = threadIdx.x;
  const size_t id = (size_t)ids[r];
  float4 *er = reinterpret_cast<float4 *>(e + (size_t)r * TH);
  if (BF16) {
    const uint4 *src = reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(emb) + id * TH);
    for (int i = t; i < TH / 8; i += 256) {
      const uint4 v = src[i];
      er[2 * i] = make_float4(bf_lo(v.x), bf_hi(v.x), bf_lo(v.y), bf_hi(v.y));
      er[2 * i + 1] = make_float4(bf_lo(v.z), bf_hi(v.z), bf_lo(v.w), bf_hi(v.w));
    }
  } else {
    const float4 *src = reinterpret_cast<const float4 *>(static_cast<const float *>(emb) + id * TH);
    for (int i = t; i < TH / 4; i += 256) er[i] = src[i];
  }
  float4 *hr = reinterpret_cast<float4 *>(h + (size_t)r * TH);
  const float4 *b1v = reinterpret_cast<const float4 *>(b1);
  for (int i = t; i < TH / 4; i += 256) hr[i] = b1v[i];
  float *yr = y + (size_t)r * ldy;
  for (int i = t; i < H; i += 256) yr[i] = b2[i];
}

// K slices of both products, at every row count: 48 ids 58 us a call (81 as full
// K on the f32 matrix cores), 520 ids 246 (339), 1100 ids 440 (552), 4000 ids
// 1490 (1520-1610). Their sums are 64 KB a row of work area, 50 us of allocation: so
// the area holds 64 rows from the start, a call beyond it runs in passes the
// first time (520 ids: 0.6 ms, 1.5-2.0 with the allocation) and the area grows at
// the second such call, up to kTextRows (2100 ids: 891 us in passes of 512 rows,
// 989 of 256, 807 in one).
constexpr int kTextSlices = 8;
constexpr int kTextRows = 1024;

// one workgroup per row: emb[ids[r]] split into operand tiles (TH % 32 == 0)
template <bool BF16>
__global__ __launch_bounds__(256) void k_text_rows_x3(const void *__restrict__ emb,
                                                      const int32_t *__restrict__ ids, int TH,
                                                      uint16_t *__restrict__ e) {
  const int r = blockIdx.x;
  const size_t id = (size_t)ids[r];
  for (int k = 8 * threadIdx.x; k < TH; k += 8 * 256) {
    float v[8];
    if (BF16) {
      const uint4 u = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(emb) + id * TH + k);
      const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; i++) v[2 * i] = bf_lo(w[i]), v[2 * i + 1] = bf_hi(w[i]);
    } else {
      const float4 *s = reinterpret_cast<const float4 *>(static_cast<const float *>(emb) + id * TH + k);
      const float4 a = s[0], b = s[1];
      v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    }
    x3_store8(e, r, k, TH, v, false);
  }
}

// 4 columns per thread: the slices' sums added in order, then to the bias
__device__ __forceinline__ void text_sum4(const float *__restrict__ part,
                                          const float *__restrict__ b, int M, int N, int m, int k,
                                          float (&v)[4]) {
  float4 p[kTextSlices];
#pragma unroll
  for (int s = 0; s < kTextSlices; s++)
    p[s] = *reinterpret_cast<const float4 *>(part + ((size_t)s * M + m) * N + k);
  const float4 bias = *reinterpret_cast<const float4 *>(b + k);
  float4 a = p[0];
#pragma unroll
  for (int s = 1; s < kTextSlices; s++) a.x += p[s].x, a.y += p[s].y, a.z += p[s].z, a.w += p[s].w;
  v[0] = bias.x + a.x, v[1] = bias.y + a.y, v[2] = bias.z + a.z, v[3] = bias.w + a.w;
}

// h = SiLU(b1 + sum), split
__global__ __launch_bounds__(256) void k_text_mid(const float *__restrict__ part,
                                                  const float *__restrict__ b1, int M, int TH,
                                                  uint16_t *__restrict__ h) {
  const int i = blockIdx.x * 256 + threadIdx.x, m = i / (TH / 4), k = 4 * (i - m * (TH / 4));
  if (m >= M) return;
  float v[4];
  text_sum4(part, b1, M, TH, m, k, v);
#pragma unroll
  for (int e = 0; e < 4; e++) v[e] = silu_clamp_f(v[e]);
  x3_store4(h, m, k, TH, v, false);
}

// y = b2 + sum
__global__ __launch_bounds__(256) void k_text_end(const float *__restrict__ part,
                                                  const float *__restrict__ b2, int M, int H,
                                                  float *__restrict__ y, int ldy) {
  const int i = blockIdx.x * 256 + threadIdx.x, m = i / (H / 4), k = 4 * (i - m * (H / 4));
  if (m >= M) return;
  float v[4];
  text_sum4(part, b2, M, H, m, k, v);
  *reinterpret_cast<float4 *>(y + (size_t)m * ldy + k) = make_float4(v[0], v[1], v[2], v[3]);
}

// w as split operand tiles instead of f32
void split_weights(Mat &w, hipStream_t st) {
  w.x3 = (uint16_t *)dev_alloc((size_t)3 * w.N * w.K * 2);
  launch_split3(w, st);
  check_hip(hipGetLastError(), "split3");
  check_hip(hipStreamSynchronize(st), "split sync");
  dev_free(w.f);
  w.f = nullptr;
}

void text_release(q3h_text_proj *t) {
  dev_free(t->emb);
  dev_free(t->fc1.f);
  dev_free(t->fc2.f);
  dev_free(t->fc1.x3);
  dev_free(t->fc2.x3);
  dev_free(t->part);
  dev_free(t->b1);
  dev_free(t->b2);
  dev_free(t->ids);
  dev_free(t->e);
  dev_free(t->h);
  dev_free(t->y);
  if (t->stream) (void)hipStreamDestroy(t->stream);
}

template <class T>
T *upload(const T *src, size_t n, const char *what) {
  require(src != nullptr, Q3H_E_ARG, std::string("q3h_text_create: ") + what + " is NULL");
  T *d = (T *)dev_alloc(sizeof(T) * n);
  check_hip(hipMemcpy(d, src, sizeof(T) * n, hipMemcpyHostToDevice), what);
  return d;
}

}  // namespace

void text_ensure(q3h_text_proj *t, int n) {
  const size_t TH = t->cfg.text_hidden, H = t->cfg.hidden;
  if (n > t->cap) {
    const int cap = std::max(n, std::max(64, 2 * t->cap));
    check_hip(hipStreamSynchronize(t->stream), "text sync");
    dev_free(t->ids);
    dev_free(t->y);
    t->ids = nullptr;
    t->y = nullptr;
    if (!t->split) {
      dev_free(t->e);
      dev_free(t->h);
      t->e = t->h = nullptr;
    }
    t->cap = 0;
    t->ids = (int32_t *)dev_alloc(sizeof(int32_t) * cap);
    t->y = (float *)dev_alloc(sizeof(float) * cap * H);
    if (!t->split) {
      t->e = (float *)dev_alloc(sizeof(float) * cap * TH);
      t->h = (float *)dev_alloc(sizeof(float) * cap * TH);
    }
    t->cap = cap;
  }
  if (!t->split || n <= t->rows || t->rows == kTextRows) return;
  if (t->rows > 0 && !t->beyond) {  // in passes of the rows there are, this once
    t->beyond = true;
    return;
  }
  const int rows = std::min(kTextRows, std::max(n, std::max(64, 2 * t->rows)));
  check_hip(hipStreamSynchronize(t->stream), "text sync");
  dev_free(t->e);
  dev_free(t->h);
  dev_free(t->part);
  t->e = t->h = t->part = nullptr;
  t->rows = 0;
  t->e = (float *)dev_alloc(x3_bytes(rows, TH));
  t->h = (float *)dev_alloc(x3_bytes(rows, TH));
  t->part = (float *)dev_alloc(sizeof(float) * kTextSlices * rows * std::max(TH, H));
  t->rows = rows;
  t->beyond = false;
}

void text_project_dev(q3h_text_proj *t, const int32_t *ids_dev, int n, float *y, int ldy,
                      hipStream_t st) {
  const q3h_text_config &c = t->cfg;
  const int TH = c.text_hidden, H = c.hidden;
  if (t->split && n > t->rows) {  // equal passes (a row's result is that of any other row count)
    const int passes = (n + t->rows - 1) / t->rows;
    for (int p = 0, r = 0; p < passes; p++) {
      const int rows = (n - r) / (passes - p);
      text_project_dev(t, ids_dev + r, rows, y + (size_t)r * ldy, ldy, st);
      r += rows;
    }
    return;
  }
  if (t->split) {
    // (the hidden rows in the memory of the embedding rows: 58.7 against 57.6 us at
    // 48 ids)
    uint16_t *e = reinterpret_cast<uint16_t *>(t->e), *h = reinterpret_cast<uint16_t *>(t->h);
    if (c.emb_dtype == Q3H_BF16)
      hipLaunchKernelGGL(k_text_rows_x3<true>, dim3(n), dim3(256), 0, st, t->emb, ids_dev, TH, e);
    else
      hipLaunchKernelGGL(k_text_rows_x3<false>, dim3(n), dim3(256), 0, st, t->emb, ids_dev, TH, e);
    auto blocks = [&](int N) { return dim3((unsigned)(((size_t)n * (N / 4) + 255) / 256)); };
    launch_gemm_x3_part(t->fc1, e, n, t->part, st, kTextSlices);
    hipLaunchKernelGGL(k_text_mid, blocks(TH), dim3(256), 0, st, t->part, t->b1, n, TH, h);
    launch_gemm_x3_part(t->fc2, h, n, t->part, st, kTextSlices);
    hipLaunchKernelGGL(k_text_end, blocks(H), dim3(256), 0, st, t->part, t->b2, n, H, y, ldy);
    check_hip(hipGetLastError(), "text projection kernels");
    return;
  }
  if (c.emb_dtype == Q3H_BF16)
    hipLaunchKernelGGL(k_text_rows<true>, dim3(n), dim3(256), 0, st, t->emb, ids_dev, TH, H,
                       t->b1, t->b2, t->e, t->h, y, ldy);
  else
    hipLaunchKernelGGL(k_text_rows<false>, dim3(n), dim3(256), 0, st, t->emb, ids_dev, TH, H,
                       t->b1, t->b2, t->e, t->h, y, ldy);
  launch_gemm_f32(t->fc1, t->e, TH, n, EPI_ADD_SILU, t->h, TH, st);
  launch_gemm_f32(t->fc2, t->h, TH, n, EPI_ADD, y, ldy, st);
  check_hip(hipGetLastError(), "text projection kernels");
}

}  // namespace q3h

using namespace q3h;

extern "C" int q3h_text_create(q3h_device *dev, const q3h_text_config *cfg, const void *emb,
                               const float *fc1_w, const float *fc1_b, const float *fc2_w,
                               const float *fc2_b, q3h_text_proj **out) {
  q3h_text_proj *t = nullptr;
  const int rc = guard([&] {
    require(dev && cfg && out, Q3H_E_ARG, "q3h_text_create: NULL argument");
    const q3h_text_config c = *cfg;
    require(c.text_vocab > 0, Q3H_E_ARG, "q3h_text_create: text_vocab must be positive");
    require(c.emb_dtype == Q3H_BF16 || c.emb_dtype == Q3H_F32, Q3H_E_ARG,
            "q3h_text_create: emb_dtype must be Q3H_BF16 or Q3H_F32");
    require(c.hidden > 0 && gemm_f32_supported(c.text_hidden, c.text_hidden) &&
                gemm_f32_supported(c.hidden, c.text_hidden),
            Q3H_E_ARG,
            "q3h_text_create: text_hidden must be 1024, 2048 or 3072 and hidden a multiple of 16");
    check_hip(hipSetDevice(dev->ordinal), "hipSetDevice");
    t = new q3h_text_proj();
    t->dev = dev;
    t->cfg = c;
    const size_t TH = c.text_hidden, H = c.hidden;
    const size_t es = c.emb_dtype == Q3H_BF16 ? 2 : 4;
    require(emb != nullptr, Q3H_E_ARG, "q3h_text_create: emb is NULL");
    t->emb = dev_alloc(es * c.text_vocab * TH);
    check_hip(hipMemcpy(t->emb, emb, es * c.text_vocab * TH, hipMemcpyHostToDevice),
              "upload text embedding");
    t->fc1.N = t->fc1.K = c.text_hidden;
    t->fc1.f = upload(fc1_w, TH * TH, "fc1_w");
    t->fc2.N = c.hidden;
    t->fc2.K = c.text_hidden;
    t->fc2.f = upload(fc2_w, H * TH, "fc2_w");
    t->b1 = upload(fc1_b, TH, "fc1_b");
    t->b2 = upload(fc2_b, H, "fc2_b");
    check_hip(hipStreamCreateWithFlags(&t->stream, hipStreamNonBlocking), "hipStreamCreate");
    // slices of whole 64-column steps, 16-byte rows
    t->split = H % 64 == 0 && TH % (64 * kTextSlices) == 0;
    if (t->split) {
      split_weights(t->fc1, t->stream);
      split_weights(t->fc2, t->stream);
    }
    text_ensure(t, 1);  // the work area of the first calls: 0.3 ms of allocations
    t->bytes = (int64_t)(es * c.text_vocab * TH + (t->split ? 6 : 4) * (TH * TH + H * TH) +
                         4 * (TH + H));
    dev->bytes += t->bytes;
    dev->stacks++;
    *out = t;
  });
  if (rc != 0 && t) {
    text_release(t);
    delete t;
  }
  return rc;
}

extern "C" int q3h_text_project(q3h_text_proj *t, const int32_t *ids, int n, float *y) {
  return guard([&] {
    require(t != nullptr, Q3H_E_ARG, "q3h_text_project: NULL projection");
    require(n >= 0, Q3H_E_ARG, "q3h_text_project: negative row count");
    if (n == 0) return;
    require(ids != nullptr && y != nullptr, Q3H_E_ARG, "q3h_text_project: NULL ids or y");
    for (int r = 0; r < n; r++)
      require(ids[r] >= 0 && ids[r] < t->cfg.text_vocab, Q3H_E_ARG,
              "q3h_text_project: text token " + std::to_string(ids[r]) + " out of range");
    std::lock_guard<std::mutex> lk(t->mu);
    check_hip(hipSetDevice(t->dev->ordinal), "hipSetDevice");
    text_ensure(t, n);
    hipStream_t st = t->stream;
    check_hip(hipMemcpyAsync(t->ids, ids, sizeof(int32_t) * n, hipMemcpyHostToDevice, st),
              "upload ids");
    text_project_dev(t, t->ids, n, t->y, t->cfg.hidden, st);
    check_hip(hipMemcpyAsync(y, t->y, sizeof(float) * n * t->cfg.hidden, hipMemcpyDeviceToHost,
                             st),
              "download y");
    check_hip(hipStreamSynchronize(st), "text sync");
  });
}

extern "C" int q3h_text_destroy(q3h_text_proj *t) {
  return guard([&] {
    if (!t) return;
    check_hip(hipSetDevice(t->dev->ordinal), "hipSetDevice");
    if (t->stream) (void)hipStreamSynchronize(t->stream);
    t->dev->bytes -= t->bytes;
    t->dev->stacks--;
    text_release(t);
    delete t;
  });
}
