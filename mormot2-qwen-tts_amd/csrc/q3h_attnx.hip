// q3h_attnx.hip - GQA attention of the int8 path (stacks with act_q8 = 1):
// a fixed evaluation order, followed to the bit by the CPU restatement of the
// same layer, and the Q8_0 quantization of its output (the o_proj input)
// fused into the epilogue. The int8 products make the layer output a
// discontinuous function of the attention output (one element on the other
// side of a rounding boundary of its block moves it by d / 127 of the block
// maximum), so this path computes every fp32 value in one documented order
// instead of to a tolerance.
//
// One workgroup per (kv head, row) for the kv head's query heads:
//  - prologue (a decode row, one new position of its own context): q, k, v
//    of the row (from the product's chunk partials, added in chunk order,
//    when the product left them as partials); RMSNorm of q and of the new k
//    (double sum of squares), RoPE as rope_pair, v copied; the first query
//    head of the kv group appends k, v to the cache, the others use their
//    own copy for the new position;
//  - scores: 16 lanes per key, lane l a fused multiply-add chain over dims
//    8l .. 8l + 7, a balanced pairwise tree over the 16 lanes (DPP row
//    operations), times 1/sqrt(128);
//  - softmax: maximum, exp_ieee(s - max), double sum, inv = (float)(1/sum),
//    weights s * inv;
//  - values: 8 chains of fused multiply-adds over the positions p = j mod 8
//    (wave w runs chain w % 8 for 128 / (waves / 8) of the dims, 512
//    coalesced bytes per key and wave), joined as ((c0 + c1) + (c2 + c3)) +
//    ((c4 + c5) + (c6 + c7));
//  - the head's 128 outputs quantized per 32-block (ggml quantize_row_q8_0_ref
//    semantics) into the operand tiles of the int8 product.
// The attention itself follows src/tts/mormot.ai.tts.qwen.lm.pas (TQwenLm.
// Forward, lm.pas:391-408) through the stack's ForwardEmbeds: causal softmax
// attention with head_dim 128, q head h reading kv head h / (heads / kv_heads).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "q3h_api_internal.h"
#include "q3h_internal.h"
#include "q3h_math.h"
#include "q3h_wave.h"

namespace q3h {
namespace {

constexpr int HD = 128;
constexpr int NCH = 8;  // value chains

template <typename KV>
__device__ __forceinline__ void load8(const KV *p, float (&o)[8]) {
  if constexpr (sizeof(KV) == 4) {
    const float4 a = reinterpret_cast<const float4 *>(p)[0];
    const float4 b = reinterpret_cast<const float4 *>(p)[1];
    o[0] = a.x, o[1] = a.y, o[2] = a.z, o[3] = a.w;
    o[4] = b.x, o[5] = b.y, o[6] = b.z, o[7] = b.w;
  } else {
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));
    const h8 v = *reinterpret_cast<const h8 *>(p);
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (float)v[e];
  }
}

template <typename KV>
__device__ __forceinline__ float2 load2(const KV *p) {
  if constexpr (sizeof(KV) == 4) {
    return *reinterpret_cast<const float2 *>(p);
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 v = *reinterpret_cast<const h2 *>(p);
    return make_float2((float)v[0], (float)v[1]);
  }
}

// elements col and col + 64 of row m: the product's output, or (nch > 0)
// its chunk partials [nch][M][ld] (nch <= kPartialSlots), loaded together
// (clamped chunk indices; qkv_sum adds the first nch in chunk order)
constexpr int NPS = kPartialSlots;
__device__ __forceinline__ void qkv_load(const float *qkv, int ld, int nch, int M, int m, int col,
                                         float (&a)[NPS], float (&b)[NPS]) {
  if (nch == 0) {
    a[0] = qkv[(size_t)m * ld + col];
    b[0] = qkv[(size_t)m * ld + col + 64];
    return;
  }
#pragma unroll
  for (int c = 0; c < NPS; c++) {
    const float *r = qkv + ((size_t)min(c, nch - 1) * M + m) * ld + col;
    a[c] = r[0];
    b[c] = r[64];
  }
}

__device__ __forceinline__ void qkv_sum(int nch, const float (&a)[NPS], const float (&b)[NPS],
                                        float &x0, float &x1) {
  if (nch == 0) {
    x0 = a[0];
    x1 = b[0];
    return;
  }
  x0 = x1 = 0.f;
#pragma unroll
  for (int c = 0; c < NPS; c++) {
    x0 = c < nch ? __fadd_rn(x0, a[c]) : x0;
    x1 = c < nch ? __fadd_rn(x1, b[c]) : x1;
  }
}

// sum over a 16-lane DPP row, the balanced pairwise tree in lane order
// ((l0 + l1) + (l2 + l3)) + ..., the same value in all 16 lanes
__device__ __forceinline__ float row16_tree(float v) {
  v = __fadd_rn(v, dpp_f<kQuadXor1>(v));
  v = __fadd_rn(v, dpp_f<kQuadXor2>(v));
  v = __fadd_rn(v, dpp_f<kHalfMirror>(v));
  v = __fadd_rn(v, dpp_f<kRowMirror>(v));
  return v;
}

// grid (kv heads, M): the GRP query heads of kv head g = blockIdx.x share one
// read of its K/V; nch > 0: the q/k/v come as nch chunk partials. SU / VU:
// the key rounds of the score loop / the positions of the value chains whose
// loads are issued together (deeper for long contexts). The first round of
// keys (and, with PV, of values) is loaded right after the q/k/v loads, so
// that it arrives during the prologue: the cache rows before the row's own
// position were written by earlier launches, and the own position's key and
// value are taken from the prologue in every round. PAIR (FUSED): rows come
// in pairs, row 2i + 1 at the position after row 2i's in the same context;
// the odd row's spare waves rebuild its pair row's key and value (the cache
// row that row 2i's workgroup writes in this launch) from row 2i's partials
// by the same code as that workgroup, so both rows run in one launch.
template <typename KV, bool FUSED, int GRP, int SU, int VU, int NT, bool PV, bool PAIR>
__global__ __launch_bounds__(NT) void k_attn_x(const RowDesc *rd, const float *qkv,
                                               const float *qkn, const float2 *rope_cs,
                                               int8_t *xq, int layer, int nch, int kvh,
                                               int M) {
  constexpr int NWV = NT / 64;
  constexpr int DPW = 16 / NWV;  // dims per lane in the value chains (2 or 1)
  // the launch shapes for contexts of several rounds take unmasked rounds
  // before the row's own position (the short-context shape keeps one code path)
  constexpr bool LONG = SU > 1;
  static_assert(NWV % NCH == 0 && DPW * 64 * (NWV / NCH) == HD, "8 chains over 128 dims");
  extern __shared__ float sc[];  // [GRP][L]: scores, then e^(score - max)
  __shared__ float qs[GRP][HD], kn[HD], vn[HD];
  __shared__ float kn2[PAIR ? HD : 1], vn2[PAIR ? HD : 1];  // the pair row's key, value
  __shared__ float cv[NCH][GRP][HD];
  __shared__ float redf[GRP][NWV];
  __shared__ double redd[GRP][NWV];
  const int g = blockIdx.x, m = blockIdx.y, t = threadIdx.x;
  const int heads = kvh * GRP, ldq = (heads + 2 * kvh) * HD;
  const int lane = t & 63, wave = t >> 6;
  const int NQ = heads * HD, nbq = NQ >> 5, mt16 = (M + 15) >> 4;
  float *dx = reinterpret_cast<float *>(xq + (size_t)mt16 * 16 * NQ);
  // output k of query head h, row m: element (m, h * 128 + k) of the operand tiles
  auto qoff = [&](int h, int k) { return qtile_offset(m, h * HD + k, mt16); };
  // vector j = wave: query head g GRP + j (j < GRP), the new k (j == GRP), v
  // (GRP + 1), and with PAIR the pair row's k and v (GRP + 2, GRP + 3, of
  // kind jv = j - 2); its loads depend on no descriptor, so they are issued
  // first, by every wave (the waves past the last vector load v again and do
  // not use it: no divergent branch before the descriptor's scalar load)
  static_assert(GRP + (PAIR ? 4 : 2) <= NWV, "one prologue vector per wave");
  const int j = wave;
  const bool pairv = PAIR && j >= GRP + 2;
  const int jv = pairv ? j - 2 : j;
  const bool odd = PAIR && (m & 1);
  const bool pj = FUSED && jv < GRP + 2;
  const int col = jv < GRP ? (g * GRP + jv) * HD : jv == GRP ? NQ + g * HD : NQ + (kvh + g) * HD;
  float pa[NPS], pb[NPS];
  if (FUSED) qkv_load(qkv, ldq, nch, M, pairv ? m & ~1 : m, col + lane, pa, pb);
  const RowDesc d = rd[m];
  if (d.pos < 0) {  // inactive row: zero blocks
    for (int i = t; i < GRP * HD; i += NT) {
      const int h = g * GRP + i / HD, k = i % HD;
      xq[qoff(h, k)] = 0;
      if ((k & 31) == 0) dx[qscale_offset(m, 4 * h + (k >> 5), nbq)] = 0.f;
    }
    return;
  }
  const int pos = d.pos, L = pos + 1;
  // positions below clean hold rows written by earlier launches (the new
  // position, and with PAIR the odd row's pair position, come from the prologue)
  const int clean = FUSED ? pos - (odd ? 1 : 0) : L;
  const size_t head_off = ((size_t)layer * kvh + g) * d.max_pos * HD;
  const KV *kc = global_ptr(reinterpret_cast<const KV *>(d.k)) + head_off;
  const KV *vc = global_ptr(reinterpret_cast<const KV *>(d.v)) + head_off;
  constexpr int KG = NT / 16;
  const int kg = t >> 4, li = t & 15;
  // value chain ch over positions ch, ch + 8, ...; dims dim0 + 64 e, e < DPW
  const int ch = wave % NCH, dim0 = (wave / NCH) * 64 + lane;

  // the first round of keys (positions u KG + kg) and values (ch + NCH u),
  // from clamped positions
  float k8p[SU][8], vp[PV ? VU : 1][DPW];
#pragma unroll
  for (int u = 0; u < SU; u++) load8(kc + (size_t)min(u * KG + kg, L - 1) * HD + 8 * li, k8p[u]);
  if constexpr (PV) {
#pragma unroll
    for (int u = 0; u < VU; u++)
#pragma unroll
      for (int e = 0; e < DPW; e++)
        vp[u][e] = (float)vc[(size_t)min(ch + NCH * u, L - 1) * HD + dim0 + 64 * e];
  }
  if (FUSED) {
    if (pj && (!pairv || odd)) {
      float x0, x1;
      qkv_sum(nch, pa, pb, x0, x1);
      if (jv <= GRP) {
        const float *w = qkn + (jv < GRP ? 0 : HD);
        const float eps = qkn[2 * HD];
        double ss = (double)x0 * (double)x0 + (double)x1 * (double)x1;
        ss = wave_sum_dpp_d(ss);
        const float inv = (float)(1.0 / sqrt(ss / HD + (double)eps));
        x0 = w[lane] * (x0 * inv);
        x1 = w[lane + 64] * (x1 * inv);
        const int rp = pairv ? max(pos - 1, 0) : pos;
        const float2 cs = rope_cs[(size_t)rp * (HD / 2) + lane];
        rope_pair(x0, x1, cs.x, cs.y);
      }
      if (jv < GRP) {
        qs[jv][lane] = x0;
        qs[jv][lane + 64] = x1;
      } else {
        const KV a0 = to_cache<KV>(x0), a1 = to_cache<KV>(x1);  // the cache's precision
        float *own = jv == GRP ? (pairv ? kn2 : kn) : (pairv ? vn2 : vn);
        own[lane] = (float)a0;
        own[lane + 64] = (float)a1;
        if (!pairv) {
          KV *dst = const_cast<KV *>(jv == GRP ? kc : vc) + (size_t)pos * HD;
          dst[lane] = a0;
          dst[lane + 64] = a1;
        }
      }
    }
  } else {
    for (int i = t; i < GRP * HD; i += NT)  // normed and rotated by the append kernel
      qs[i / HD][i % HD] = qkv[(size_t)m * ldq + (g * GRP + i / HD) * HD + i % HD];
  }
  __syncthreads();

  // scores: key group kg = t / 16 takes positions kg, kg + 32, ...; the loads
  // of SU positions are issued together
  const float scale = (float)(1.0 / __builtin_sqrt((double)HD));
  {
    float qv[GRP][8], kn8[8], kp8[8];
#pragma unroll
    for (int j = 0; j < GRP; j++)
#pragma unroll
      for (int e = 0; e < 8; e++) qv[j][e] = qs[j][8 * li + e];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      kn8[e] = FUSED ? kn[8 * li + e] : 0.f;
      kp8[e] = PAIR ? kn2[8 * li + e] : 0.f;
    }
    for (int p0 = 0; p0 < L; p0 += KG * SU) {
      // unconditional loads from clamped positions (a guarded load would be
      // waited for on its own), then the new position's own k, zeros past L
      float k8[SU][8];
      if (p0 == 0) {
#pragma unroll
        for (int u = 0; u < SU; u++)
#pragma unroll
          for (int e = 0; e < 8; e++) k8[u][e] = k8p[u][e];
      } else {
#pragma unroll
        for (int u = 0; u < SU; u++)
          load8(kc + (size_t)min(p0 + u * KG + kg, L - 1) * HD + 8 * li, k8[u]);
      }
      // a round wholly before the row's own position needs no masks
      auto round = [&](auto masked) {
        constexpr bool MK = decltype(masked)::value;
        if constexpr (MK) {
#pragma unroll
          for (int u = 0; u < SU; u++) {
            const int p = p0 + u * KG + kg;
#pragma unroll
            for (int e = 0; e < 8; e++)
              k8[u][e] = p >= L               ? 0.f
                         : FUSED && p == pos   ? kn8[e]
                         : odd && p == pos - 1 ? kp8[e]
                                               : k8[u][e];
          }
        }
#pragma unroll
        for (int u = 0; u < SU; u++) {
          const int p = p0 + u * KG + kg;
#pragma unroll
          for (int j = 0; j < GRP; j++) {
            float a = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) a = fmaf(qv[j][e], k8[u][e], a);
            a = row16_tree(a);
            if ((!MK || p < L) && li == 0) sc[j * L + p] = __fmul_rn(a, scale);
          }
        }
      };
      if (LONG && p0 + KG * SU <= clean)
        round(std::false_type{});
      else
        round(std::true_type{});
    }
  }
  __syncthreads();

  // softmax per head
  float inv[GRP], ew[GRP];
  if constexpr (!LONG) {
    // the one-round shape (covers of at most 32 positions): one wave holds a
    // head's scores, one per lane, so every wave takes the maximum, the
    // exponentials and the double sum itself (no barrier, no LDS trip) and
    // keeps its lane's exponential for the value weights
#pragma unroll
    for (int j = 0; j < GRP; j++) {
      const float sv = lane < L ? sc[j * L + lane] : -INFINITY;
      const float mx = wave_max_dpp(sv);
      ew[j] = lane < L ? exp_ieee(__fsub_rn(sv, mx)) : 0.f;
      inv[j] = (float)(1.0 / wave_sum_dpp_d((double)ew[j]));
    }
  } else {
#pragma unroll
    for (int j = 0; j < GRP; j++) ew[j] = 0.f;
    float mx[GRP];
#pragma unroll
    for (int j = 0; j < GRP; j++) mx[j] = -INFINITY;
    for (int p = t; p < L; p += NT)
#pragma unroll
      for (int j = 0; j < GRP; j++) mx[j] = fmaxf(mx[j], sc[j * L + p]);
#pragma unroll
    for (int j = 0; j < GRP; j++) {
      mx[j] = wave_max_dpp(mx[j]);
      if (lane == 0) redf[j][wave] = mx[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < GRP; j++) {
      float v = redf[j][0];
#pragma unroll
      for (int w = 1; w < NWV; w++) v = fmaxf(v, redf[j][w]);
      mx[j] = v;
    }
    double sum[GRP];
#pragma unroll
    for (int j = 0; j < GRP; j++) sum[j] = 0.0;
    for (int p = t; p < L; p += NT)
#pragma unroll
      for (int j = 0; j < GRP; j++) {
        const float e = exp_ieee(__fsub_rn(sc[j * L + p], mx[j]));
        sc[j * L + p] = e;
        sum[j] += (double)e;
      }
#pragma unroll
    for (int j = 0; j < GRP; j++) {
      sum[j] = wave_sum_dpp_d(sum[j]);
      if (lane == 0) redd[j][wave] = sum[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < GRP; j++) {
      double s2 = 0.0;
#pragma unroll
      for (int w = 0; w < NWV; w++) s2 += redd[j][w];
      inv[j] = (float)(1.0 / s2);
    }
  }

  // values: chain ch = wave % 8 over positions p = ch mod 8, dims dim0 + 64 e,
  // every head of the group; the loads of VU positions issued together
  {
    float c[DPW][GRP];
#pragma unroll
    for (int e = 0; e < DPW; e++)
#pragma unroll
      for (int j = 0; j < GRP; j++) c[e][j] = 0.f;
    float vnd[DPW], vpd[DPW];
#pragma unroll
    for (int e = 0; e < DPW; e++) {
      vnd[e] = FUSED ? vn[dim0 + 64 * e] : 0.f;
      vpd[e] = PAIR ? vn2[dim0 + 64 * e] : 0.f;
    }
    for (int p0 = ch; p0 < L; p0 += NCH * VU) {
      float v[VU][DPW];
      if (PV && p0 == ch) {
#pragma unroll
        for (int u = 0; u < VU; u++)
#pragma unroll
          for (int e = 0; e < DPW; e++) v[u][e] = vp[PV ? u : 0][e];
      } else {
#pragma unroll
        for (int u = 0; u < VU; u++)
#pragma unroll
          for (int e = 0; e < DPW; e++)
            v[u][e] = (float)vc[(size_t)min(p0 + NCH * u, L - 1) * HD + dim0 + 64 * e];
      }
      // the new position: its own v; past L: zero (the clamped load may have
      // read the new row before it was written); weights of the round read
      // together, past L a zero weight times a zero value adds an exact zero to
      // the chain. A round wholly before the row's own position needs no masks.
      auto round = [&](auto masked) {
        constexpr bool MK = decltype(masked)::value;
        if constexpr (MK) {
#pragma unroll
          for (int u = 0; u < VU; u++) {
            const int p = p0 + NCH * u;
#pragma unroll
            for (int e = 0; e < DPW; e++)
              v[u][e] = p >= L               ? 0.f
                        : FUSED && p == pos   ? vnd[e]
                        : odd && p == pos - 1 ? vpd[e]
                                              : v[u][e];
          }
        }
        float wgt[VU][GRP];
#pragma unroll
        for (int u = 0; u < VU; u++) {
          const int p = p0 + NCH * u;  // the same for the whole wave
#pragma unroll
          for (int j = 0; j < GRP; j++) {
            const float e = LONG ? sc[j * L + (MK ? min(p, L - 1) : p)] : lane_f(ew[j], min(p, L - 1));
            wgt[u][j] = !MK || p < L ? __fmul_rn(e, inv[j]) : 0.f;
          }
        }
#pragma unroll
        for (int u = 0; u < VU; u++)
#pragma unroll
          for (int j = 0; j < GRP; j++)
#pragma unroll
            for (int e = 0; e < DPW; e++) c[e][j] = fmaf(wgt[u][j], v[u][e], c[e][j]);
      };
      if (LONG && p0 + NCH * (VU - 1) < clean)
        round(std::false_type{});
      else
        round(std::true_type{});
    }
#pragma unroll
    for (int j = 0; j < GRP; j++)
#pragma unroll
      for (int e = 0; e < DPW; e++) cv[ch][j][dim0 + 64 * e] = c[e][j];
  }
  __syncthreads();

  // quantize each head's 128 outputs per 32-block (a 32-lane half-wave each)
  for (int i = t; i < GRP * HD; i += NT) {
    const int j = i / HD, k = i % HD, h = g * GRP + j;
    const float o = __fadd_rn(
        __fadd_rn(__fadd_rn(cv[0][j][k], cv[1][j][k]), __fadd_rn(cv[2][j][k], cv[3][j][k])),
        __fadd_rn(__fadd_rn(cv[4][j][k], cv[5][j][k]), __fadd_rn(cv[6][j][k], cv[7][j][k])));
    float amax = fabsf(o);
    amax = half_max_dpp(amax);
    const float dq = __fdiv_rn(amax, 127.0f);
    const float id = dq != 0.f ? __fdiv_rn(1.0f, dq) : 0.f;
    xq[qoff(h, k)] = (int8_t)(int)roundf(__fmul_rn(o, id));
    if ((k & 31) == 0) dx[qscale_offset(m, 4 * h + (k >> 5), nbq)] = (float)(_Float16)dq;
  }
}

// four cached values as floats
template <typename KV>
__device__ __forceinline__ float4 load4(const KV *p) {
  if constexpr (sizeof(KV) == 4) {
    return *reinterpret_cast<const float4 *>(p);
  } else {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const h4 h = *reinterpret_cast<const h4 *>(p);
    return make_float4((float)h[0], (float)h[1], (float)h[2], (float)h[3]);
  }
}

// Two chains of 8 fused multiply-adds (the first product rounded alone, as the
// multiply-add onto zero does) of the 16 elements of q, held one per lane of
// every 16-lane row, and the lane's own k: a0 over elements 0 .. 7, a1 over 8
// .. 15. The element is taken from the row by the multiply-add itself (DPP
// row_newbcast), an operand form the compiler does not build for fused
// multiply-adds; the wait states let a q written just before be read by DPP.
__device__ __forceinline__ void dot8x2(float q, const float4 &k0, const float4 &k1,
                                       const float4 &k2, const float4 &k3, float &a0, float &a1) {
#define Q3H_BC(n) " row_newbcast:" #n " row_mask:0xf bank_mask:0xf\n"
  asm("s_nop 1\n"
      "v_mul_f32_dpp %0, %2, %3" Q3H_BC(0) "v_mul_f32_dpp %1, %2, %11" Q3H_BC(8)
      "v_fmac_f32_dpp %0, %2, %4" Q3H_BC(1) "v_fmac_f32_dpp %1, %2, %12" Q3H_BC(9)
      "v_fmac_f32_dpp %0, %2, %5" Q3H_BC(2) "v_fmac_f32_dpp %1, %2, %13" Q3H_BC(10)
      "v_fmac_f32_dpp %0, %2, %6" Q3H_BC(3) "v_fmac_f32_dpp %1, %2, %14" Q3H_BC(11)
      "v_fmac_f32_dpp %0, %2, %7" Q3H_BC(4) "v_fmac_f32_dpp %1, %2, %15" Q3H_BC(12)
      "v_fmac_f32_dpp %0, %2, %8" Q3H_BC(5) "v_fmac_f32_dpp %1, %2, %16" Q3H_BC(13)
      "v_fmac_f32_dpp %0, %2, %9" Q3H_BC(6) "v_fmac_f32_dpp %1, %2, %17" Q3H_BC(14)
      "v_fmac_f32_dpp %0, %2, %10" Q3H_BC(7) "v_fmac_f32_dpp %1, %2, %18" Q3H_BC(15)
      : "=&v"(a0), "=&v"(a1)
      : "v"(q), "v"(k0.x), "v"(k0.y), "v"(k0.z), "v"(k0.w), "v"(k1.x), "v"(k1.y), "v"(k1.z),
        "v"(k1.w), "v"(k2.x), "v"(k2.y), "v"(k2.z), "v"(k2.w), "v"(k3.x), "v"(k3.y), "v"(k3.z),
        "v"(k3.w));
#undef Q3H_BC
}

// The same attention for prompt rows (q normed and rotated, every K/V row of
// the tile's context already appended), several rows sharing one read of the
// keys and values: a workgroup of 4 waves per (kv head, tile of R = PAIRS / GRP
// consecutive positions of one context), PAIRS (row, query head) pairs, every
// value by the operations of k_attn_x in the same order.
//  - scores: 64 keys at a time through LDS, then a key per lane in 128
//    registers; the wave's PAIRS / 4 pairs one after another, the query's
//    elements broadcast by DPP: 16 chains of 8 fused multiply-adds and the 15
//    adds of their tree in one lane, where k_attn_x's 16 lanes per key pay 4
//    DPP adds each (146 instructions per 64 keys and pair against about 200)
//    and re-read the key from L2 for every row;
//  - softmax: the wave's pairs together, a position per lane; the weights e * inv left in place of the scores;
//  - values: half-wave 2 wave + h runs chain 2 wave + h over positions = chain
//    mod 8, 4 dims per lane, all pairs (the value row loaded once for them, the
//    weights of a position as 16-byte LDS broadcasts); positions after a row's
//    own are skipped by selects, in the tile's last rounds only;
//  - the chains joined through LDS 8 pairs at a time and quantized.
// Scores in LDS: [position][PAIRS + 4] (rows of 16-byte multiples whose lanes
// start 4 banks apart). What bounds it is the VALU: about 4.3 instructions per
// (row, head, position).
template <typename KV, int GRP, int PAIRS>
__global__ __launch_bounds__(256, 2) void k_attn_xp(const RowDesc *__restrict__ rd,
                                                    const float *__restrict__ qkv,
                                                    int8_t *__restrict__ xq, int layer, int kvh,
                                                    int M, const int2 *__restrict__ tiles) {
  constexpr int R = PAIRS / GRP, ST = PAIRS + 4, PW = PAIRS / 4, KS = HD + 4;
  static_assert(PAIRS % 8 == 0 && PAIRS % GRP == 0, "8 pairs per join round");
  extern __shared__ float sm[];
  float *ks = sm;             // [64][KS] keys; then the joining sums [4][8][HD]
  float *sc = sm + 64 * KS;   // [positions rounded up to 64][ST]
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = blockIdx.x, heads = kvh * GRP, ldq = (heads + 2 * kvh) * HD;
  const int NQ = heads * HD, nbq = NQ >> 5, mt16 = (M + 15) >> 4;
  const int tl = gridDim.y - 1 - blockIdx.y;
  const int2 tile = tiles ? tiles[blockIdx.y] : make_int2(tl * R, min(R, M - tl * R));
  const int q0 = tile.x, nq = tile.y;
  const RowDesc d = rd[q0];
  const int pos0 = d.pos, L = pos0 + nq;  // positions of the tile's last row
  const size_t head_off = ((size_t)layer * kvh + g) * d.max_pos * HD;
  const KV *kc = global_ptr(reinterpret_cast<const KV *>(d.k)) + head_off;
  const KV *vc = global_ptr(reinterpret_cast<const KV *>(d.v)) + head_off;
  const float scale = (float)(1.0 / __builtin_sqrt((double)HD));

  // scores
  float4 kn[8];
  auto load_keys = [&](int kb) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int f = t + 256 * i;  // float4 f of the block's 64 x 32
      kn[i] = load4(kc + (size_t)min(kb + (f >> 5), L - 1) * HD + 4 * (f & 31));
    }
  };
  // element 16 k + lane % 16 of the query of the wave's pair i, k < 8
  float qn[8];
  auto load_q = [&](int i) {
    const int pair = wave * PW + i, r = min(pair / GRP, nq - 1);
    const float *q = qkv + (size_t)(q0 + r) * ldq + (g * GRP + pair % GRP) * HD + (lane & 15);
#pragma unroll
    for (int k = 0; k < 8; k++) qn[k] = q[16 * k];
  };
  load_keys(0);
  load_q(0);
  for (int kb = 0; kb < L; kb += 64) {
    if (kb) __syncthreads();  // the waves have read the block before
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int f = t + 256 * i;
      *reinterpret_cast<float4 *>(&ks[(f >> 5) * KS + 4 * (f & 31)]) = kn[i];
    }
    __syncthreads();
    float4 kr[HD / 4];
#pragma unroll
    for (int i = 0; i < HD / 4; i++) kr[i] = *reinterpret_cast<const float4 *>(&ks[lane * KS + 4 * i]);
    load_keys(kb + 64);
    for (int i = 0; i < PW; i++) {
      const int pair = wave * PW + i, r = min(pair / GRP, nq - 1);
      float q[8];
#pragma unroll
      for (int k = 0; k < 8; k++) q[k] = qn[k];
      load_q(i + 1 < PW ? i + 1 : 0);
      if (kb > pos0 + r) continue;  // wholly after the row
      float a[16];
#pragma unroll
      for (int k = 0; k < 8; k++)
        dot8x2(q[k], kr[4 * k], kr[4 * k + 1], kr[4 * k + 2], kr[4 * k + 3], a[2 * k], a[2 * k + 1]);
#pragma unroll
      for (int n = 8; n >= 1; n >>= 1)
#pragma unroll
        for (int c = 0; c < n; c++) a[c] = __fadd_rn(a[2 * c], a[2 * c + 1]);
      sc[(kb + lane) * ST + pair] = __fmul_rn(a[0], scale);
    }
  }
  __syncthreads();

  // softmax: the wave's PW pairs together, a position per lane and round
  {
    float mx[PW], inv[PW];
    double sum[PW];
    int Lr[PW];
    float *sw = sc + wave * PW;
#pragma unroll
    for (int i = 0; i < PW; i++) {
      Lr[i] = pos0 + min((wave * PW + i) / GRP, nq - 1) + 1;
      mx[i] = -INFINITY;
      sum[i] = 0.0;
    }
    auto get = [&](int p, float (&v)[PW]) {
#pragma unroll
      for (int i = 0; i < PW; i += 2) {
        const float2 u = *reinterpret_cast<const float2 *>(&sw[p * ST + i]);
        v[i] = u.x;
        v[i + 1] = u.y;
      }
    };
    auto put = [&](int p, const float (&v)[PW]) {
#pragma unroll
      for (int i = 0; i < PW; i += 2)
        *reinterpret_cast<float2 *>(&sw[p * ST + i]) = make_float2(v[i], v[i + 1]);
    };
    float v[PW];
    for (int p = lane; p < L; p += 64) {
      get(p, v);
#pragma unroll
      for (int i = 0; i < PW; i++) mx[i] = p < Lr[i] ? fmaxf(mx[i], v[i]) : mx[i];
    }
#pragma unroll
    for (int i = 0; i < PW; i++) mx[i] = wave_max_dpp(mx[i]);
    for (int p = lane; p < L; p += 64) {
      get(p, v);
#pragma unroll
      for (int i = 0; i < PW; i++) {
        v[i] = exp_ieee(__fsub_rn(v[i], mx[i]));
        sum[i] += p < Lr[i] ? (double)v[i] : 0.0;
      }
      put(p, v);
    }
#pragma unroll
    for (int i = 0; i < PW; i++) inv[i] = (float)(1.0 / wave_sum_dpp_d(sum[i]));
    for (int p = lane; p < L; p += 64) {
      get(p, v);
#pragma unroll
      for (int i = 0; i < PW; i++) v[i] = __fmul_rn(v[i], inv[i]);
      put(p, v);
    }
  }
  __syncthreads();

  // values
  const int ch = 2 * wave + (lane >> 5), dim = 4 * (lane & 31);
  float c[PAIRS][4];
#pragma unroll
  for (int j = 0; j < PAIRS; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) c[j][e] = 0.f;
  auto load_v = [&](int p) { return load4(vc + (size_t)min(p, L - 1) * HD + dim); };
  // position p of the chain, for every pair (MASK: those whose row is at p or after)
  auto step = [&](int p, const float4 &v, auto masked) {
    constexpr bool MASK = decltype(masked)::value;
    const float *w = sc + (size_t)(MASK ? min(p, L - 1) : p) * ST;
#pragma unroll
    for (int j0 = 0; j0 < PAIRS; j0 += 4) {
      const float4 w4 = *reinterpret_cast<const float4 *>(w + j0);
      const float wj[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        float *cj = c[j0 + j];
        const bool on = !MASK || p <= pos0 + (j0 + j) / GRP;
        cj[0] = on ? fmaf(wj[j], v.x, cj[0]) : cj[0];
        cj[1] = on ? fmaf(wj[j], v.y, cj[1]) : cj[1];
        cj[2] = on ? fmaf(wj[j], v.z, cj[2]) : cj[2];
        cj[3] = on ? fmaf(wj[j], v.w, cj[3]) : cj[3];
      }
    }
  };
  int p0 = 0;
  float4 vb[4];
#pragma unroll
  for (int u = 0; u < 4; u++) vb[u] = load_v(ch + 8 * u);
  for (; p0 + 31 <= pos0; p0 += 32) {
    float4 vn[4];
#pragma unroll
    for (int u = 0; u < 4; u++) vn[u] = load_v(p0 + 32 + ch + 8 * u);
#pragma unroll
    for (int u = 0; u < 4; u++) step(p0 + ch + 8 * u, vb[u], std::false_type{});
#pragma unroll
    for (int u = 0; u < 4; u++) vb[u] = vn[u];
  }
  for (; p0 < L; p0 += 8) {
    const float4 v = load_v(p0 + ch);
    step(p0 + ch, v, std::true_type{});
  }
  // the sums of chains 2 wave and 2 wave + 1 added across the halves, the
  // waves' through LDS 8 pairs at a time, quantized per 32-block (8 lanes x 4
  // dims): thread t takes pair t / 32 of the 8, dims 4 (t % 32) .. + 3
  float *dx = reinterpret_cast<float *>(xq + (size_t)mt16 * 16 * NQ);
#pragma unroll
  for (int j0 = 0; j0 < PAIRS; j0 += 8) {
    __syncthreads();  // the keys, or the sums of the round before, are read
    // the lower half holds pair j0 + i, the upper one pair j0 + 4 + i
    const int half = lane >> 5;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      float4 o;
      o.x = swap32_add(c[j0 + i][0], c[j0 + 4 + i][0]);
      o.y = swap32_add(c[j0 + i][1], c[j0 + 4 + i][1]);
      o.z = swap32_add(c[j0 + i][2], c[j0 + 4 + i][2]);
      o.w = swap32_add(c[j0 + i][3], c[j0 + 4 + i][3]);
      *reinterpret_cast<float4 *>(&ks[(wave * 8 + 4 * half + i) * HD + dim]) = o;
    }
    __syncthreads();
    const int jp = t >> 5, k = 4 * (t & 31), pair = j0 + jp, r = pair / GRP;
    float o[4], amax = 0.f;
    float4 s4[4];
#pragma unroll
    for (int w = 0; w < 4; w++) s4[w] = *reinterpret_cast<const float4 *>(&ks[(w * 8 + jp) * HD + k]);
    const float sv[4][4] = {{s4[0].x, s4[0].y, s4[0].z, s4[0].w},
                            {s4[1].x, s4[1].y, s4[1].z, s4[1].w},
                            {s4[2].x, s4[2].y, s4[2].z, s4[2].w},
                            {s4[3].x, s4[3].y, s4[3].z, s4[3].w}};
#pragma unroll
    for (int e = 0; e < 4; e++) {
      o[e] = __fadd_rn(__fadd_rn(sv[0][e], sv[1][e]), __fadd_rn(sv[2][e], sv[3][e]));
      amax = fmaxf(amax, fabsf(o[e]));
    }
    amax = quad_max_dpp(amax);
    amax = fmaxf(amax, dpp_f_keep<kHalfMirror>(amax));
    if (r < nq) {
      const float dq = __fdiv_rn(amax, 127.0f);
      const float id = dq != 0.f ? __fdiv_rn(1.0f, dq) : 0.f;
      unsigned packed = 0;
#pragma unroll
      for (int e = 0; e < 4; e++)
        packed |= (unsigned)(uint8_t)(int8_t)(int)roundf(__fmul_rn(o[e], id)) << (8 * e);
      const int m = q0 + r, h = g * GRP + pair % GRP;
      *reinterpret_cast<unsigned *>(xq + qtile_offset(m, h * HD + k, mt16)) = packed;
      if ((t & 7) == 0) dx[qscale_offset(m, 4 * h + (k >> 5), nbq)] = (float)(_Float16)dq;
    }
  }
}

}  // namespace

bool attn_x_supported(int heads, int kvh, int head_dim, int max_positions) {
  return head_dim == HD && kvh > 0 && heads % kvh == 0 &&
         (heads / kvh == 1 || heads / kvh == 2 || heads / kvh == 4) && max_positions > 0 &&
         (size_t)max_positions * (heads / kvh) <= (size_t)kAttnXMaxPositions;
}

template <typename KV, bool F, int SU, int VU, int NT, bool PV, bool PAIR = false>
void attn_x_grp(const AttnArgs &a, int M, int nch, const QAct &xa, int max_positions,
                hipStream_t st) {
  const dim3 grid(a.kvh, M);
  const int grp = a.heads / a.kvh;
  // the kernel takes the q/k/v row stride as (heads + 2 kv heads) * 128, so
  // that its arguments fit the 14 dwords preloaded in SGPRs (the grid size,
  // a hidden argument past them, would be a dependent load before the first)
  require(a.ldq == (a.heads + 2 * a.kvh) * HD, Q3H_E_ARG, "attention: q/k/v rows not packed");
  const size_t lds = sizeof(float) * (size_t)grp * max_positions;
#define Q3H_ATTNX(G)                                                                         \
  hipLaunchKernelGGL((k_attn_x<KV, F, G, SU, VU, NT, PV, PAIR>), grid, dim3(NT), lds, st, a.rd, \
                     a.qkv, a.qkn, a.rope_cs, xa.q, a.layer, nch, a.kvh, M)
  if (grp == 1)
    Q3H_ATTNX(1);
  else if (grp == 2)
    Q3H_ATTNX(2);
  else
    Q3H_ATTNX(4);
#undef Q3H_ATTNX
}

// short contexts (the code predictor's 16 positions): one round of each loop;
// decode rows over longer contexts: 128 keys and 64 values per round, the
// first values loaded with the keys (the loads of a round come from clamped
// positions, so deeper rounds cost a short context their full width: 1024
// threads with 512 keys and 128 values per round measured 2.5 us slower per
// talker layer over 32 ragged contexts); prefill rows 256 keys and 128 values
// per round. Results do not depend on the thread count or the round depths.
template <typename KV, bool F>
void attn_x_len(const AttnArgs &a, int M, int nch, const QAct &xa, int max_positions,
                bool pairs, hipStream_t st) {
  if (F && pairs)  // the short shape only (attn_x_pairs_supported)
    attn_x_grp<KV, F, 1, 4, 512, true, true>(a, M, nch, xa, max_positions, st);
  else if (max_positions <= 32)
    attn_x_grp<KV, F, 1, 4, 512, true>(a, M, nch, xa, max_positions, st);
  else if constexpr (F)
    attn_x_grp<KV, F, 4, 8, 512, true>(a, M, nch, xa, max_positions, st);
  else
    attn_x_grp<KV, F, 8, 16, 512, false>(a, M, nch, xa, max_positions, st);
}

// LDS of k_attn_xp: the keys, then a score row per position
template <int PAIRS>
constexpr size_t attn_xp_lds(int positions) {
  return sizeof(float) * (64 * (HD + 4) + (size_t)((positions + 63) / 64 * 64) * (PAIRS + 4));
}
constexpr size_t kLdsBytes = 160 << 10;

// The rows of k_attn_xp's tiles, 0 where k_attn_x takes the rows: 16 (row,
// head) pairs per workgroup where that still makes 1024 workgroups, 8 below
// (601 rows: 51 us against 71; 1201 rows: 224 with 16, 275 with 8), and where
// 16 pairs' scores do not fit in LDS (above 1600 positions; 2300 rows: 870
// against 1016 us by k_attn_x). k_attn_x takes contexts above 2688 positions
// (8 pairs' scores do not fit), and few rows onto a long context, whose walk
// over the keys it spreads over more workgroups. 3798 rows of 32 prompts: 110
// us, 430 by k_attn_x; 203 rows 13.5 / 29; 70 rows 7.9 / 12.9; 17 rows 5.7 /
// 6.7.
int attn_x_tile_rows(int heads, int kvh, int M, int positions) {
  const int grp = heads / kvh;
  if (M < 8 || 4 * M < positions || attn_xp_lds<8>(positions) > kLdsBytes) return 0;
  const int r16 = 16 / grp;
  return (M + r16 - 1) / r16 * kvh >= 1024 && attn_xp_lds<16>(positions) <= kLdsBytes ? r16 : 8 / grp;
}

template <typename KV, int GRP, int PAIRS>
void attn_xp_launch(const AttnArgs &a, int M, int positions, const QAct &xa, hipStream_t st) {
  constexpr int R = PAIRS / GRP;
  const dim3 grid(a.kvh, a.tiles ? a.n_tiles : (M + R - 1) / R);
  const size_t lds = attn_xp_lds<PAIRS>(positions);
  if (lds > (64 << 10))
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_attn_xp<KV, GRP, PAIRS>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes),
              "attention LDS");
  hipLaunchKernelGGL((k_attn_xp<KV, GRP, PAIRS>), grid, dim3(256), lds, st, a.rd, a.qkv, xa.q,
                     a.layer, a.kvh, M, a.tiles);
}

template <typename KV, int GRP>
void attn_xp_grp(const AttnArgs &a, int M, int rows, int positions, const QAct &xa,
                 hipStream_t st) {
  if (rows == 16 / GRP)
    attn_xp_launch<KV, GRP, 16>(a, M, positions, xa, st);
  else
    attn_xp_launch<KV, GRP, 8>(a, M, positions, xa, st);
}

bool launch_attn_x_prompt(const AttnArgs &a, int M, int positions, bool kv16, const QAct &xa,
                          hipStream_t st) {
  const int rows = a.tiles ? a.tile_rows : attn_x_tile_rows(a.heads, a.kvh, M, positions);
  if (rows == 0) return false;
  require(a.ldq == (a.heads + 2 * a.kvh) * HD, Q3H_E_ARG, "attention: q/k/v rows not packed");
  const int grp = a.heads / a.kvh;
#define Q3H_XP(KV)                                             \
  do {                                                         \
    if (grp == 1)                                              \
      attn_xp_grp<KV, 1>(a, M, rows, positions, xa, st);       \
    else if (grp == 2)                                         \
      attn_xp_grp<KV, 2>(a, M, rows, positions, xa, st);       \
    else                                                       \
      attn_xp_grp<KV, 4>(a, M, rows, positions, xa, st);       \
  } while (0)
  if (kv16)
    Q3H_XP(_Float16);
  else
    Q3H_XP(float);
#undef Q3H_XP
  return true;
}

bool attn_x_pairs_supported(int max_positions) { return max_positions <= 32; }

void launch_attn_x(const AttnArgs &a, int M, bool fused, bool kv16, int qkv_chunks,
                   const QAct &xa, int max_positions, hipStream_t st, bool pairs) {
  const int nch = fused ? qkv_chunks : 0;
  require(!pairs || (fused && M % 2 == 0 && attn_x_pairs_supported(max_positions)), Q3H_E_ARG,
          "attention: row pairs need the fused short-context shape and an even row count");
  if (kv16) {
    if (fused)
      attn_x_len<_Float16, true>(a, M, nch, xa, max_positions, pairs, st);
    else
      attn_x_len<_Float16, false>(a, M, nch, xa, max_positions, false, st);
  } else {
    if (fused)
      attn_x_len<float, true>(a, M, nch, xa, max_positions, pairs, st);
    else
      attn_x_len<float, false>(a, M, nch, xa, max_positions, false, st);
  }
}

}  // namespace q3h
