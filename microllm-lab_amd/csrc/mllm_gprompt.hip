// mllm_gprompt.hip -- batched prompts (infer.js:553-577 forwardPrompt) for the
// models of the kind-generic step (mllm_generic.hip): a chunk of T prompt
// tokens goes through every layer as five kernels (GPT-2: seven) instead of
// token by token, so a matrix is read once per 32 tokens and the launches of
// a prompt do not grow with its length.
//
// GEMMs on the bf16 matrix cores at float32 accuracy: the activations are
// three bf16 planes (mllm_planes.h, exact), the weights one, two or three
// (gp_planes), and these products are formed: x0 w0, x1 w0, x2 w0 (1 plane),
// + x0 w1, x1 w1 (2), + x0 w2 (3).  What one plane leaves of a value is at most
// 2^-8 of it, two planes 2^-17, so each product left out (x2 w1, with 3 planes
// x1 w2 too) is at most 2^-25 of x w: half a float32 rounding.  Q8 group-32 and Q4 weights are
// the de-quantised values rounded to float32 (the token steps multiply the
// integers and scale the sums).  x0 w0 has an accumulator of its own, the
// corrections share another, added at the end, so the roundings of the large
// sum are one per 16 columns.
//
// No kernel needs a whole row except the norms' statistics, so nothing but the
// GEMMs and the attention is launched for a llama layer:
//   QKV    y = r_t (W (x g)): planes of x g from the kernel that formed x,
//          r_t = 1 / sqrt(mean x^2 + eps) from that kernel's per-64-column
//          sums; epilogue RoPE, q, K and V to the cache
//   ATTN   causal attention in float32, its output written as planes
//   O      x += W_o o; planes of x g2 and the sums of squares of x
//   UP     gate and up rows of the same units: silu(g) u as planes
//   DOWN   x += W_2 h; planes of x g1' (the next layer's norm) and the sums
// GPT-2's LayerNorm subtracts a mean first, which would cancel in the scaled
// form, so its rows are normalised by a kernel of their own.
//
// What bounds it: at a few hundred tokens a launch has fewer wave tiles than
// the chip has SIMDs, and its time is latency: 2.5-3 us until the first
// operands arrive (they come from HBM or another XCD's L2), as much again for
// each further round of loads, about 1 us for a cold instruction cache.  So a
// wave tile is 64 rows x 32 tokens; a workgroup is 1 to 8 waves that take
// slices of the columns (added in order through LDS), about 1024 waves a
// launch; a wave loads 5 half-groups (of 16 columns) ahead; what the epilogue
// reads is loaded first; the XCDs are laid out so that their L2s fetch least.
// Measured at 200 tokens of the 135M shape in f16, us a launch: QKV 14.0 ->
// 8.7 (whole groups ahead, read past the slice's end; epilogue loads after the
// products, eight values a thread), O and down 13.3 -> 11.6, gate/up 14.0 ->
// 12.3; the prompt 2.27 -> 2.03 ms.  Weights loaded with the non-temporal
// policy were slower (2.40 ms): other token tiles read them again.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "mllm_device.h"
#include "mllm_generic.h"
#include "mllm_gprompt.h"
#include "mllm_host.h"
#include "mllm_kinds.h"
#include "mllm_planes.h"

namespace mllm {
namespace {

typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

enum { GP_QKV = 0, GP_RESID = 1, GP_SWIGLU = 2, GP_GELU = 3 };
constexpr int GPHD = 64;
constexpr int GPW = 8;               // waves (column slices) of a GEMM workgroup at most
constexpr int GPT = 32 * 68;         // floats of one slice's tile in LDS: 32 tokens x 64 rows (+ 4)

struct GpGemm {
  const uint8_t *w0, *w1;   // tiled rows of sub-tile 0 and 1 (32 rows each)
  const float *s0, *s1;     // per-row scales, or null
  int off1;                 // row tile of sub-tile 1 minus that of sub-tile 0
  int rstep;                // row tiles of the matrix per workgroup (2; 1 where w1 is another matrix)
  int ng;                   // groups per row
  int rtiles, ttiles;       // row tiles of rstep, token tiles
  int xt, nbx;              // token groups of XCDs; row tiles per XCD
  int n, tt0, li, pos0;     // tokens, first token tile, layer, first position
  const uint8_t *px;        // the input's planes
  uint8_t *po;              // the output's planes, or null
  int ldp;                  // groups per token of po
  const float *bias;        // per row, or null
  const float *gain;        // RESID: the next norm's gains (po = planes of x gain), or null
  int rms;                  // the input is x g: scale by 1 / sqrt(mean x^2 + eps)
};

// A half (16 columns) of a group: the token tile's planes, two row tiles' planes.
template <int NP>
struct GpLd {
  v8b x[3], w[2][NP];
};

__device__ __forceinline__ v8b ld_op(const uint8_t *p) {
  return __builtin_bit_cast(v8b, *reinterpret_cast<const uint4 *>(p));
}

__device__ __forceinline__ v16f mfma(v8b a, v8b b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// One sub-tile: hi += w0 x0, lo += the corrections.
template <int NP>
__device__ __forceinline__ void gp_half(const v8b (&x)[3], const v8b (&w)[NP], v16f &hi, v16f &lo) {
  hi = mfma(w[0], x[0], hi);
  lo = mfma(w[0], x[1], lo);
  lo = mfma(w[0], x[2], lo);
  if constexpr (NP > 1) {
    lo = mfma(w[1], x[0], lo);
    lo = mfma(w[1], x[1], lo);
  }
  if constexpr (NP > 2) lo = mfma(w[2], x[0], lo);
}

// What an epilogue item (four rows of one token) reads from memory.  A thread
// of an eight-slice workgroup has one item and loads it before its operands:
// loaded after the products it would cost the launch a second memory latency.
struct GpItem {
  float4 s0, bias;  // the rows' scales and biases
  float4 a, b;      // RESID: residual, next gains; QKV: cos, sin; SWIGLU: b = the up rows' scales
};

__device__ __forceinline__ float el(const float4 &v, int e) { return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w; }

template <int EPI>
__device__ __forceinline__ GpItem gp_item(const GpArgs &A, const GpGemm &G, int rt, int rd, int t, int c) {
  GpItem I;
  const int row = 32 * rt + 4 * c;
  I.s0 = I.bias = I.a = I.b = make_float4(0.f, 0.f, 0.f, 0.f);
  if (G.s0) I.s0 = ld4u(G.s0 + row);
  if (EPI == GP_SWIGLU && G.s1) I.b = ld4u(G.s1 + row);
  if (G.bias) I.bias = ld4u(G.bias + row);
  t = min(t, G.n - 1);
  if (EPI == GP_RESID) {
    I.a = *reinterpret_cast<const float4 *>(A.x + (size_t)t * A.D + row);
    if (G.gain) I.b = ld4u(G.gain + row);
  }
  if (EPI == GP_QKV && 4 * c < rd) {
    const size_t at = (size_t)(G.pos0 + t) * rd;
    float cs[4], sn[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      cs[e] = A.rope_cos[at + min(4 * c + e, rd - 1)];
      sn[e] = A.rope_sin[at + min(4 * c + e, rd - 1)];
    }
    I.a = make_float4(cs[0], cs[1], cs[2], cs[3]);
    I.b = make_float4(sn[0], sn[1], sn[2], sn[3]);
  }
  return I;
}

// Dynamic LDS: blockDim / 64 tiles of GPT floats, then 32 norm scales.
template <int EPI, int NP>
__global__ __launch_bounds__(64 * GPW) void k_gp_gemm(GpArgs A, GpGemm G) {
  extern __shared__ __attribute__((aligned(16))) float buf[];
  const int KS = blockDim.x >> 6, ks = tid() >> 6, lane = tid() & 63, j = lane & 31, hh = lane >> 5;
  // workgroup b runs on XCD b % 8, each with an L2 of its own: the XCDs are a
  // grid of G.xt token groups x 8 / G.xt row groups (launch_gemm)
  const int xr = 8 / G.xt, xcd = blockIdx.x & 7, kb = blockIdx.x >> 3;
  const int bx = xcd % xr + xr * (kb % G.nbx), by = xcd / xr + G.xt * (kb / G.nbx);
  if (bx >= G.rtiles || by >= G.ttiles) return;
  const int T0 = (G.tt0 + by) * 32, rt = bx * G.rstep;
  const int ng = G.ng, hb = 2 * ng * ks / KS, he = 2 * ng * (ks + 1) / KS;  // this wave's halves
  const uint8_t *wa = G.w0 + (size_t)rt * ng * NP * 2048 + 16 * lane;
  const uint8_t *wb = G.w1 + (size_t)(rt + G.off1) * ng * NP * 2048 + 16 * lane;
  const uint8_t *xa = G.px + (size_t)(G.tt0 + by) * ng * BPX + 16 * lane;
  auto load = [&](int h) {
    GpLd<NP> L;
    const int g = h >> 1, m = h & 1;
#pragma unroll
    for (int p = 0; p < 3; ++p) L.x[p] = ld_op(xa + (size_t)g * BPX + (2 * p + m) * 1024);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      L.w[0][p] = ld_op(wa + ((size_t)g * NP + p) * 2048 + m * 1024);
      L.w[1][p] = ld_op(wb + ((size_t)g * NP + p) * 2048 + m * 1024);
    }
    return L;
  };
  // first the epilogue's loads and the residual's sums of squares (eight lanes
  // a token), then the operands': loads complete in order
  constexpr int CH = EPI == GP_SWIGLU ? 8 : 16;
  const int rd = EPI == GP_QKV && A.arch == 0 && (rt >> 1) < A.NH + A.NKV ? A.rope_dim : 0;
  const GpItem first = gp_item<EPI>(A, G, rt, rd, T0 + (int)tid() / CH, tid() % CH);
  const int nb = A.D >> 6;
  float s0 = 0.f, s1 = 0.f;
  if (G.rms && tid() < 256) {
    const float *sp = A.ss + (size_t)(T0 + (tid() >> 3)) * nb;
    const int b = tid() & 7;
    if (b < nb) s0 = sp[b];
    if (b + 8 < nb) s1 = sp[b + 8];
  }
  constexpr int RD = NP == 1 ? 7 : NP == 2 ? 5 : 4;  // halves of loads in flight: as many as the registers hold
  GpLd<NP> ring[RD];
#pragma unroll
  for (int i = 0; i < RD; ++i) ring[i] = load(min(hb + i, he - 1));
  float *rs = buf + KS * GPT;
  if (G.rms) {
    for (int i = tid(); i < 256; i += blockDim.x) {
      const float *sp = A.ss + (size_t)(T0 + (i >> 3)) * nb;
      float s = 0.f;
      if (i == (int)tid()) {
        s = s0 + s1;
        for (int b = (i & 7) + 16; b < nb; b += 8) s += sp[b];
      } else {
        for (int b = i & 7; b < nb; b += 8) s += sp[b];
      }
      s = sum8f(s);
      if ((i & 7) == 0) rs[i >> 3] = 1.0f / sqrtf(s / (float)A.D + A.eps);
    }
  }
  v16f h0, h1, l0, l1;
#pragma unroll
  for (int v = 0; v < 16; ++v) h0[v] = h1[v] = l0[v] = l1[v] = 0.f;
  for (int h = hb; h < he; h += RD)
#pragma unroll
    for (int i = 0; i < RD; ++i) {
      if (h + i >= he) break;
      gp_half<NP>(ring[i].x, ring[i].w[0], h0, l0);
      gp_half<NP>(ring[i].x, ring[i].w[1], h1, l1);
      if (h + i + RD < he) ring[i] = load(h + i + RD);
    }
  // an infinity or NaN among the operands is in hi as it is, in lo as NaN
  float big = 0.f;
#pragma unroll
  for (int v = 0; v < 16; ++v) big = __builtin_elementwise_maximum(__builtin_elementwise_maximum(big, fabsf(l0[v])), fabsf(l1[v]));
  if (__any(!(big < INFINITY))) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      l0[v] = fabsf(h0[v]) < INFINITY ? l0[v] : 0.f;
      l1[v] = fabsf(h1[v]) < INFINITY ? l1[v] : 0.f;
    }
  }
  // value v of lane (j, hh): token j, row 8 (v / 4) + 4 hh + v % 4
  float *mine = buf + ks * GPT + j * 68 + 4 * hh;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    *reinterpret_cast<float4 *>(mine + 8 * q) = make_float4(h0[4 * q] + l0[4 * q], h0[4 * q + 1] + l0[4 * q + 1],
                                                            h0[4 * q + 2] + l0[4 * q + 2], h0[4 * q + 3] + l0[4 * q + 3]);
    *reinterpret_cast<float4 *>(mine + 32 + 8 * q) = make_float4(h1[4 * q] + l1[4 * q], h1[4 * q + 1] + l1[4 * q + 1],
                                                                 h1[4 * q + 2] + l1[4 * q + 2], h1[4 * q + 3] + l1[4 * q + 3]);
  }
  __syncthreads();
  if (KS > 1) {
    for (int i = tid(); i < 512; i += blockDim.x) {
      float *p = buf + (i >> 4) * 68 + 4 * (i & 15);
      float4 o[GPW];
#pragma unroll
      for (int k = 0; k < GPW; ++k) o[k] = *reinterpret_cast<const float4 *>(p + (k < KS ? k : 0) * GPT);
      float4 s = o[0];
#pragma unroll
      for (int k = 1; k < GPW; ++k)
        if (k < KS) s = make_float4(s.x + o[k].x, s.y + o[k].y, s.z + o[k].z, s.w + o[k].w);
      *reinterpret_cast<float4 *>(p) = s;
    }
    __syncthreads();
  }
  // epilogue: item = (token jt, rows 4c .. 4c+3 of the tile).  Four values a
  // thread keep the code short: a launch runs it once, from a cold
  // instruction cache.
  for (int it = tid(); it < 32 * CH; it += blockDim.x) {
    const int jt = it / CH, c = it % CH, t = T0 + jt;
    const bool in = t < G.n;
    const float *row = buf + jt * 68;
    const float r = G.rms ? rs[jt] : 1.f;
    const GpItem I = it == (int)tid() ? first : gp_item<EPI>(A, G, rt, rd, t, c);
    // output e of the item
    auto at = [&](int e) {
      float v = row[4 * c + e] * r;
      if (G.s0) v *= el(I.s0, e);
      return G.bias ? v + el(I.bias, e) : v;
    };
    float y[4];
    if (EPI == GP_QKV) {
      if (!in) continue;
      const int head = rt >> 1, pos = G.pos0 + t, half = rd >> 1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = 4 * c + e;
        y[e] = at(e);
        if (d < rd) {  // rotate-half RoPE on the first rd components (infer.js:208-225)
          const int m = d < half ? d + half : d - half;
          float o = row[m] * r;
          if (G.s0) o *= G.s0[32 * rt + m];
          y[e] = __builtin_fmaf(y[e], el(I.a, e), (d < half ? -o : o) * el(I.b, e));
        }
      }
      if (head < A.NH) {
        *reinterpret_cast<float4 *>(A.q + (size_t)t * A.D + head * GPHD + 4 * c) = make_float4(y[0], y[1], y[2], y[3]);
      } else {
        const bool is_k = head < A.NH + A.NKV;
        const int kvh = is_k ? head - A.NH : head - A.NH - A.NKV;
        const size_t k = ((((size_t)G.li * 2 + (is_k ? 0 : 1)) * A.NKV + kvh) * A.max_seq + pos) * GPHD + 4 * c;
        if (A.kv_fp16) {
          // the cache holds the float32 value rounded: not formed in one rounding
#pragma unroll
          for (int e = 0; e < 4; ++e) asm("" : "+v"(y[e]));
          const __half2 a = __floats2half2_rn(y[0], y[1]), b = __floats2half2_rn(y[2], y[3]);
          *reinterpret_cast<uint2 *>(reinterpret_cast<__half *>(A.kv) + k) =
              make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
        } else {
          *reinterpret_cast<float4 *>(reinterpret_cast<float *>(A.kv) + k) = make_float4(y[0], y[1], y[2], y[3]);
        }
      }
    } else if (EPI == GP_RESID) {
      float sq = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[e] = el(I.a, e) + at(e);
        sq += y[e] * y[e];
      }
      sq = row16_sum(sq);  // the token's 64 columns of this tile
      if (!in) continue;
      *reinterpret_cast<float4 *>(A.x + (size_t)t * A.D + 32 * rt + 4 * c) = make_float4(y[0], y[1], y[2], y[3]);
      if (G.gain) {
        if (c == 0) A.ss[(size_t)t * (A.D >> 6) + (rt >> 1)] = sq;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] *= el(I.b, e);
        planes_store4(G.po + ((size_t)(T0 >> 5) * G.ldp + rt) * BPX, jt, c, y);
      }
    } else {
      if (!in) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (EPI == GP_SWIGLU) {
          const float a = at(e);
          float b = row[32 + 4 * c + e] * r;
          if (G.s1) b *= el(I.b, e);
          y[e] = (a / (1.0f + expf(-a))) * b;  // infer.js:175-181
        } else {
          const float v = at(e);
          y[e] = 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));  // infer.js:166-172
        }
      }
      planes_store4(G.po + ((size_t)(T0 >> 5) * G.ldp + rt) * BPX, jt, c, y);
    }
  }
}

// Columns 8c .. 8c+7 of a token.
__device__ __forceinline__ void planes_put8(uint8_t *tile, int j, int c, const float (&v)[8]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float u[4] = {v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]};
    planes_store4(tile, j, 2 * c + h, u);
  }
}

// The tokens' embedding rows (infer.js:360-420) and, for llama, the first
// norm's input: planes of x g and the sums of squares.
__global__ __launch_bounds__(WG) void k_gp_embed(GpArgs A, const float *gain, int pos0) {
  const int t = blockIdx.x, D = A.D, nc = D >> 3, id = A.ids[t];
  const GMat &W = A.emb;
  const bool quant = W.kind == MLLM_Q8 || W.kind == MLLM_Q8G32 || W.kind == MLLM_Q4;
  const int pos = min(pos0 + t, A.max_seq - 1);
  for (int c0 = 0; c0 < nc; c0 += WG) {
    const int c = min(c0 + (int)tid(), nc - 1);
    const bool in = c0 + (int)tid() < nc;
    float v[8], sq = 0.f;
    const float sc = load8(W, id, c, v), rs = W.kind == MLLM_Q8 ? W.s[id] : sc;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (quant) v[e] *= rs;
      if (A.arch == 1) {
        if (quant && A.sf) v[e] /= A.sf[8 * c + e];
        v[e] += A.wpe[(size_t)pos * D + 8 * c + e];
      }
      sq += v[e] * v[e];
    }
    sq = sum8f(sq);
    if (!in) continue;
    float4 *x = reinterpret_cast<float4 *>(A.x + (size_t)t * D + 8 * c);
    x[0] = make_float4(v[0], v[1], v[2], v[3]);
    x[1] = make_float4(v[4], v[5], v[6], v[7]);
    if (gain) {
      if ((c & 7) == 0) A.ss[(size_t)t * (D >> 6) + (c >> 3)] = sq;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= gain[8 * c + e];
      planes_put8(A.pxa + (size_t)(t >> 5) * (D >> 5) * BPX, t & 31, c, v);
    }
  }
}

// GPT-2: LayerNorm (infer.js:147-164) of tokens t0 .. n-1, one wave each, as
// planes.
__global__ __launch_bounds__(WG) void k_gp_ln(GpArgs A, const float *g, int t0, int n) {
  const int t = t0 + (int)blockIdx.x * (WG / 64) + (tid() >> 6), lane = tid() & 63, D = A.D;
  if (t >= n) return;  // uniform in the wave
  const float *x = A.x + (size_t)t * D;
  float s = 0.f;
  for (int i = lane; i < D; i += 64) s += x[i];
  const float mean = wave_sum(s) / (float)D;
  s = 0.f;
  for (int i = lane; i < D; i += 64) {
    const float d = x[i] - mean;
    s += d * d;
  }
  const float r = 1.0f / sqrtf(wave_sum(s) / (float)D + 1e-5f);
  for (int c = lane; c < (D >> 3); c += 64) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (x[8 * c + e] - mean) * r * g[8 * c + e] + g[D + 8 * c + e];
    planes_put8(A.pxa + (size_t)(t >> 5) * (D >> 5) * BPX, t & 31, c, v);
  }
}

// ---------------------------------------------------------------- attention
// Workgroup (32-query tile, query head), its 32-key blocks dealt round-robin to
// GAS waves.  Per block, on the float32 matrix cores:
//   S^T = K Q^T    v_mfma_f32_32x32x2_f32, A = the keys (lane: key j), B = the
//                  queries; step (c, e) takes dimensions 8c + e and 8c + 4 + e
//   O^T += V^T P^T A = the values (lane: dimension j), B = the weights straight
//                  from the S^T registers: value v of lane half hh is key
//                  8 (v / 4) + 4 hh + v % 4
// so that a lane holds one query's scores and outputs, and a wave needs no LDS
// until the end, where the waves' (outputs, max, sum) meet, in wave order, a
// thread per four outputs.
//
// Float32 operands, sums, softmax weights and exponentials throughout, as in
// k_g_attn: keys, values and queries of any magnitude keep their 24 bits.
// (Halves of f16 pairs, as the Q4 prompts take them, end at 65504 and lose bits
// below 2^-13.)
//
// What bounds it: 64 MFMAs of 64 cycles a block, from about 1000 tokens on, with
// 400 VALU instructions of softmax between them and two waves on a SIMD; below,
// the launch and one latency per eight blocks.  At 2000 tokens of the 135M shape
// 72 us a launch (64 TFLOP/s over the unmasked half): 116 with a clamp and a
// 64-bit address per load, instead of resources that end after the last row, and
// the heads of a tile apart in the grid.  The f16-pair kernel, whose units have
// sixteen times the rate, took 16.0 us at 200 tokens (now 9.4), at 28 and 77 of
// 11 heads with an f16 cache 7.1 and 7.3 (6.4 and 6.8), at 196 of 7 heads with an
// f16 cache 9.4 (10.1); prompts of 1000 tokens 3.85 ms (3.18), 2000 6.41 (5.55)
// and with an f16 cache 4.81 (5.66).
constexpr int GAS = 8;

// Cache elements as loaded, four components of a key (k) and one of a value
// (v) at byte `off` of a head's rows; past the rows of the resource: 0.
template <bool F16>
struct KvRaw;
template <>
struct KvRaw<false> {
  typedef float4 K;
  typedef float V;
  static __device__ __forceinline__ K k(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(K, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  }
  static __device__ __forceinline__ V v(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  }
  static __device__ __forceinline__ float4 k4(const K &r) { return r; }
  static __device__ __forceinline__ float f(V r) { return r; }
};
template <>
struct KvRaw<true> {
  typedef uint2 K;
  typedef unsigned short V;
  static __device__ __forceinline__ K k(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(K, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  }
  static __device__ __forceinline__ V v(__amdgpu_buffer_rsrc_t r, int off) {
    return (V)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
  }
  static __device__ __forceinline__ float4 k4(const K &r) {
    return make_float4(f16_bits(r.x & 0xffffu), f16_bits(r.x >> 16), f16_bits(r.y & 0xffffu), f16_bits(r.y >> 16));
  }
  static __device__ __forceinline__ float f(V r) { return f16_bits(r); }
};
constexpr size_t kAttnLds = sizeof(float) * GAS * (GPT + 64);

__device__ __forceinline__ v16f mfma_f32(float a, float b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ bool finite(float v) { return fabsf(v) < INFINITY; }

// ND: halves of the output's 64 dimensions that a workgroup forms (blockIdx.z:
// which, if one).
template <bool F16, int ND>
__global__ __launch_bounds__(64 * GAS) void k_gp_attn(GpArgs A, int li, int n, int pos0, int tt0) {
  extern __shared__ __attribute__((aligned(16))) float buf[];  // [GAS][GPT] outputs, [GAS][2][32] (max, sum)
  const int T0 = (tt0 + (int)(gridDim.y - 1 - blockIdx.y)) * 32;  // the longest tiles first
  const int hq = blockIdx.x, kvh = hq / (A.NH / A.NKV), d0 = ND == 1 ? 32 * (int)blockIdx.z : 0;
  const int wv = __builtin_amdgcn_readfirstlane(tid() >> 6), lane = tid() & 63, j = lane & 31, hh = lane >> 5;
  const int qpos = pos0 + T0 + j, qlast = pos0 + min(T0 + 32, n) - 1;  // last key any query of the tile sees
  const int nb = (qlast >> 5) + 1, used = min(nb, GAS);
  constexpr int ES = F16 ? 2 : 4, ROW = ES * GPHD;  // bytes of an element, of a row
  const size_t hb = (size_t)A.max_seq * ROW;         // of a head
  uint8_t *kp = static_cast<uint8_t *>(A.kv) + ((size_t)li * 2 * A.NKV + kvh) * hb;
  // resources that end after row qlast: what the last block reads past it is 0
  const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc(kp, (short)0, (qlast + 1) * ROW, 0x00020000);
  const __amdgpu_buffer_rsrc_t vres =
      __builtin_amdgcn_make_buffer_rsrc(kp + A.NKV * hb, (short)0, (qlast + 1) * ROW, 0x00020000);
  float4 q[8];
  typename KvRaw<F16>::K kr[8];
  typename KvRaw<F16>::V vr[ND][16];
  auto load_k = [&](int b) {
    const int at = (32 * b + j) * ROW + 4 * hh * ES;
#pragma unroll
    for (int c = 0; c < 8; ++c) kr[c] = KvRaw<F16>::k(kres, at + 8 * c * ES);
  };
  auto load_v = [&](int b) {
    const int at = (32 * b + 4 * hh) * ROW + (d0 + j) * ES;
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
      for (int d = 0; d < ND; ++d) vr[d][v] = KvRaw<F16>::v(vres, at + (8 * (v >> 2) + (v & 3)) * ROW + 32 * d * ES);
  };
  {
    const float *qr = A.q + (size_t)min(T0 + j, n - 1) * A.D + hq * GPHD + 4 * hh;
#pragma unroll
    for (int c = 0; c < 8; ++c) q[c] = *reinterpret_cast<const float4 *>(qr + 8 * c);
  }
  if (wv < nb) {
    load_k(wv);
    load_v(wv);
  }
  float m = -INFINITY, l = 0.f;
  v16f o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[d][v] = 0.f;
  for (int b = wv; b < nb; b += GAS) {
    v16f s;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float4 k = KvRaw<F16>::k4(kr[c]);
      s = mfma_f32(k.x, q[c].x, s);
      s = mfma_f32(k.y, q[c].y, s);
      s = mfma_f32(k.z, q[c].z, s);
      s = mfma_f32(k.w, q[c].w, s);
    }
    if (b + GAS < nb) load_k(b + GAS);
    const bool masked = 32 * b + 31 > pos0 + T0;  // the block reaches past a query of the tile
    float mx = m;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] *= A.attn_scale;
      if (masked && 32 * b + 8 * (v >> 2) + 4 * hh + (v & 3) > qpos) s[v] = -INFINITY;
      mx = fmaxf(mx, s[v]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float ref = score_ref(mx), alpha = expf(m - ref);
    float ps = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = expf(s[v] - ref);
      ps += s[v];
    }
    l = l * alpha + (ps + __shfl_xor(ps, 32));
    if (__any(mx != m)) {
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[d][v] *= alpha;
    }
    m = mx;
    bool whole = true;
    if (masked) {
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v) whole &= finite(KvRaw<F16>::f(vr[d][v]));
    }
    if (__all(whole)) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int d = 0; d < ND; ++d) o[d] = mfma_f32(KvRaw<F16>::f(vr[d][v]), s[v], o[d]);
    } else {
      // An infinity or NaN among the values of a block with masked keys: their
      // weight is 0 and 0 times it NaN, in the rows of queries that do not see
      // it.  It is left out of the products, and counted for the queries that
      // do: those are NaN.
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        v16f hit;
#pragma unroll
        for (int v = 0; v < 16; ++v) hit[v] = 0.f;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const float val = KvRaw<F16>::f(vr[d][v]);
          const bool sees = 32 * b + 8 * (v >> 2) + 4 * hh + (v & 3) <= qpos;
          o[d] = mfma_f32(finite(val) ? val : 0.f, s[v], o[d]);
          hit = mfma_f32(finite(val) ? 0.f : 1.f, sees ? 1.f : 0.f, hit);
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) o[d][v] = hit[v] > 0.f ? NAN : o[d][v];
      }
    }
    if (b + GAS < nb) load_v(b + GAS);
  }
  // value v of lane (j, hh): query j, dimension 8 (v / 4) + 4 hh + v % 4 of either half
  float *ml = buf + GAS * GPT;
  if (wv < used) {
    float *mine = buf + wv * GPT + j * 68 + 4 * hh;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4 *>(mine + 32 * d + 8 * g) =
            make_float4(o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]);
    ml[wv * 64 + 32 * hh + j] = hh ? l : m;
  }
  __syncthreads();
  const int jt = (int)tid() / (8 * ND), c = (int)tid() % (8 * ND);
  if (jt >= 32 || T0 + jt >= n) return;
  float M = -INFINITY;
  for (int w = 0; w < used; ++w) M = fmaxf(M, ml[w * 64 + jt]);
  M = score_ref(M);
  float L = 0.f, r[4] = {0.f, 0.f, 0.f, 0.f};
  for (int w = 0; w < used; ++w) {
    const float f = expf(ml[w * 64 + jt] - M);
    const float4 u = *reinterpret_cast<const float4 *>(buf + w * GPT + jt * 68 + 4 * c);
    L = __builtin_fmaf(ml[w * 64 + 32 + jt], f, L);
    r[0] = __builtin_fmaf(u.x, f, r[0]), r[1] = __builtin_fmaf(u.y, f, r[1]);
    r[2] = __builtin_fmaf(u.z, f, r[2]), r[3] = __builtin_fmaf(u.w, f, r[3]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = r[e] / L;
  planes_store4(A.pxo + ((size_t)(T0 >> 5) * (A.D >> 5) + 2 * hq) * BPX, jt, (d0 >> 2) + c, r);
}

// Thread = one lane's 16 bytes of every plane: eight columns of one row.
__global__ __launch_bounds__(WG) void k_gp_tile(GMat W, int np, uint8_t *dst) {
  const int ng = W.cols >> 5;
  const size_t units = (size_t)(W.rows >> 5) * ng * 128;  // (row tile, group, half, lane)
  for (size_t u = (size_t)blockIdx.x * WG + tid(); u < units; u += (size_t)gridDim.x * WG) {
    const int l = (int)(u & 127);  // half l / 64, lane l % 64
    const size_t tg = u >> 7;
    const int g = (int)(tg % ng), r = (int)(tg / ng) * 32 + (l & 31);
    float v[8];
    const float sc = load8(W, r, 4 * g + 2 * (l >> 6) + ((l >> 5) & 1), v);
    uint32_t p[4][3];
#pragma unroll
    for (int e = 0; e < 4; ++e) bf16_split2(v[2 * e] * sc, v[2 * e + 1] * sc, p[e]);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (k < np)
        *reinterpret_cast<uint4 *>(dst + (tg * np + k) * 2048 + 16 * l) = make_uint4(p[0][k], p[1][k], p[2][k], p[3][k]);
  }
}

// ---------------------------------------------------------------- host
typedef void (*GpKernel)(GpArgs, GpGemm);
const GpKernel kGpKernels[4][3] = {
    {k_gp_gemm<GP_QKV, 1>, k_gp_gemm<GP_QKV, 2>, k_gp_gemm<GP_QKV, 3>},
    {k_gp_gemm<GP_RESID, 1>, k_gp_gemm<GP_RESID, 2>, k_gp_gemm<GP_RESID, 3>},
    {k_gp_gemm<GP_SWIGLU, 1>, k_gp_gemm<GP_SWIGLU, 2>, k_gp_gemm<GP_SWIGLU, 3>},
    {k_gp_gemm<GP_GELU, 1>, k_gp_gemm<GP_GELU, 2>, k_gp_gemm<GP_GELU, 3>},
};
void (*const kGpAttn[2][2])(GpArgs, int, int, int, int) = {{k_gp_attn<false, 1>, k_gp_attn<false, 2>},
                                                           {k_gp_attn<true, 1>, k_gp_attn<true, 2>}};
// Workgroups (32-token tiles times heads) up to which the output's halves are
// apart: while both fit the 256 CUs, a block's 64 MFMAs become 48 for each (the
// scores are formed twice).  9 heads, 200 tokens: 10.9 -> 9.4 us a launch; 7
// heads, 196 tokens 11.5 -> 10.1.
constexpr int kAttnHalves = 128;
size_t gp_lds(int ks) { return sizeof(float) * ((size_t)ks * GPT + 32); }

// Column slices per tile: doubled while the launch has fewer than 1024 waves
// and every slice keeps two groups.
// XCDs: with xt token groups and 8 / xt row groups each XCD's L2 fetches a part
// of the weights and a part of the planes, xt times the weights' bytes plus
// 8 / xt times the planes' in all; the split that fetches least.
void launch_gemm(int epi, const GpArgs &A, const GpMat &W, GpGemm G, hipStream_t s) {
  G.rtiles = W.rows / (32 * G.rstep);
  G.ttiles = (G.n + 31) / 32 - G.tt0;
  int ks = 1;
  while (ks < GPW && G.rtiles * G.ttiles * ks < 1024 && G.ng / (2 * ks) >= 2) ks *= 2;
  const long wb = (long)G.rtiles * 64 * W.np * 2, xb = (long)G.ttiles * 32 * 6;  // bytes per column
  G.xt = 1;
  for (int xt = 2; xt <= 8; xt *= 2)
    if (xt * wb + 8 / xt * xb < G.xt * wb + 8 / G.xt * xb) G.xt = xt;
  const int xr = 8 / G.xt, nby = (G.ttiles + G.xt - 1) / G.xt;
  G.nbx = (G.rtiles + xr - 1) / xr;
  hipLaunchKernelGGL(kGpKernels[epi][W.np - 1], dim3(8 * G.nbx * nby), dim3(64 * ks), gp_lds(ks), s, A, G);
}

GpGemm gemm_of(const GpMat &W, int n, int tt0, const uint8_t *px) {
  GpGemm G{};
  G.w0 = G.w1 = W.t;
  G.s0 = G.s1 = W.rs;
  G.off1 = 1;
  G.rstep = 2;
  G.ng = W.cols >> 5;
  G.n = n;
  G.tt0 = tt0;
  G.px = px;
  return G;
}

}  // namespace

int gp_planes(int kind) { return kind == MLLM_BF16 || kind == MLLM_Q8 ? 1 : kind == MLLM_F16 ? 2 : 3; }

size_t gp_tiled_bytes(int rows, int cols, int np) {
  return (size_t)(rows >> 5) * (cols >> 5) * np * 2048;
}

int gp_tile(const GMat &W, int np, void *dst, GpMat *out, hipStream_t s) {
  MLLM_CHECK(W.rows % 32 == 0 && W.cols % 32 == 0, "matrix %d x %d cannot be tiled", W.rows, W.cols);
  const size_t units = (size_t)(W.rows / 32) * (W.cols / 32) * 128;
  hipLaunchKernelGGL(k_gp_tile, dim3((unsigned)std::min<size_t>((units + WG - 1) / WG, 8192)), dim3(WG), 0, s, W, np,
                     static_cast<uint8_t *>(dst));
  MLLM_HIP(hipGetLastError());
  *out = GpMat{static_cast<uint8_t *>(dst), W.kind == MLLM_Q8 ? W.s : nullptr, W.rows, W.cols, np};
  return 0;
}

bool gp_supported(const GpArgs &A) {
  return A.D == A.NH * GPHD && A.NH % A.NKV == 0 && A.NH / A.NKV <= 4 && A.FF % 64 == 0;
}

namespace {
size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }
size_t px_bytes(int tc, int cols) { return al256((size_t)((tc + 31) / 32) * (cols >> 5) * BPX); }
}  // namespace

size_t gp_buffer_bytes(const GpArgs &A, int tc) {
  const size_t tp = (size_t)((tc + 31) / 32) * 32;  // the scales of a whole tile are read
  return al256(sizeof(int32_t) * tc) + 2 * al256(sizeof(float) * tc * A.D) + al256(sizeof(float) * tp * (A.D >> 6)) +
         2 * px_bytes(tc, A.D) + px_bytes(tc, A.FF);
}

void gp_carve(GpArgs &A, void *base, int tc) {
  const size_t tp = (size_t)((tc + 31) / 32) * 32;
  uint8_t *p = static_cast<uint8_t *>(base);
  auto take = [&](size_t b) {
    uint8_t *q = p;
    p += b;
    return q;
  };
  A.tc = tc;
  A.ids = reinterpret_cast<int32_t *>(take(al256(sizeof(int32_t) * tc)));
  A.x = reinterpret_cast<float *>(take(al256(sizeof(float) * tc * A.D)));
  A.q = reinterpret_cast<float *>(take(al256(sizeof(float) * tc * A.D)));
  A.ss = reinterpret_cast<float *>(take(al256(sizeof(float) * tp * (A.D >> 6))));
  A.pxa = take(px_bytes(tc, A.D));
  A.pxo = take(px_bytes(tc, A.D));
  A.pxh = take(px_bytes(tc, A.FF));
}

int gp_init() {
  for (const auto &row : kGpKernels)
    for (GpKernel k : row)
      MLLM_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)gp_lds(GPW)));
  for (const auto &row : kGpAttn)
    for (const auto k : row)
      MLLM_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kAttnLds));
  return 0;
}

int gp_layers(const GpArgs &A, const int32_t *ids, int n, int pos0, bool last, const float **row, hipStream_t s) {
  MLLM_CHECK(n > 0 && n <= A.tc && pos0 >= 0 && pos0 + n <= A.max_seq, "prompt chunk of %d tokens at %d out of range", n,
             pos0);
  MLLM_HIP(hipMemcpyAsync(A.ids, ids, sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
  const bool gpt2 = A.arch == 1;
  const int ntt = (n + 31) / 32, ngd = A.D >> 5;
  hipLaunchKernelGGL(k_gp_embed, dim3(n), dim3(WG), 0, s, A, gpt2 ? nullptr : A.layers[0].n1, pos0);
  auto ln = [&](const float *g, int t0) {
    hipLaunchKernelGGL(k_gp_ln, dim3((n - t0 + WG / 64 - 1) / (WG / 64)), dim3(WG), 0, s, A, g, t0, n);
  };
  for (int li = 0; li < A.L; ++li) {
    const GpLayer &W = A.layers[li];
    const bool final_layer = li == A.L - 1;
    if (gpt2) ln(W.n1, 0);
    GpGemm Q = gemm_of(W.qkv, n, 0, A.pxa);
    Q.li = li;
    Q.pos0 = pos0;
    Q.bias = gpt2 ? W.qkv_b : nullptr;
    Q.rms = !gpt2;
    launch_gemm(GP_QKV, A, W.qkv, Q, s);
    if (final_layer && !last) break;
    // the prompt's last token needs its own tile of the last layer only
    const int tt0 = final_layer ? ntt - 1 : 0;
    const int nd = A.NH * (ntt - tt0) <= kAttnHalves ? 1 : 2;
    hipLaunchKernelGGL(kGpAttn[A.kv_fp16 ? 1 : 0][nd - 1], dim3(A.NH, ntt - tt0, 2 / nd), dim3(64 * GAS), kAttnLds, s, A, li,
                       n, pos0, tt0);
    GpGemm O = gemm_of(W.proj, n, tt0, A.pxo);
    O.bias = gpt2 ? W.proj_b : nullptr;
    O.gain = gpt2 ? nullptr : W.n2;
    O.po = A.pxa;
    O.ldp = ngd;
    launch_gemm(GP_RESID, A, W.proj, O, s);
    if (gpt2) ln(W.n2, 32 * tt0);
    GpGemm U = gemm_of(W.w1, n, tt0, A.pxa);
    U.po = A.pxh;
    U.ldp = A.FF >> 5;
    U.rms = !gpt2;
    if (gpt2) {
      U.bias = W.fc_b;
      launch_gemm(GP_GELU, A, W.w1, U, s);
    } else {
      U.w1 = W.w3.t;
      U.s1 = W.w3.rs;
      U.off1 = 0;
      U.rstep = 1;
      launch_gemm(GP_SWIGLU, A, W.w1, U, s);
    }
    GpGemm Dn = gemm_of(W.w2, n, tt0, A.pxh);
    Dn.bias = gpt2 ? W.mproj_b : nullptr;
    Dn.gain = gpt2 || final_layer ? nullptr : A.layers[li + 1].n1;
    Dn.po = A.pxa;
    Dn.ldp = ngd;
    launch_gemm(GP_RESID, A, W.w2, Dn, s);
  }
  MLLM_HIP(hipGetLastError());
  if (row) *row = A.x + (size_t)(n - 1) * A.D;
  return 0;
}

}  // namespace mllm
