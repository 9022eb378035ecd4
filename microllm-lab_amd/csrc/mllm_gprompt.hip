// mllm_gprompt.hip -- batched prompts (infer.js:553-577 forwardPrompt) for the
// models of the kind-generic step (mllm_generic.hip): a chunk of T prompt
// tokens goes through every layer as five kernels (GPT-2: seven) instead of
// token by token, so a matrix is read once per 32 tokens and the launches of
// a prompt do not grow with its length.
//
// GEMMs on the bf16 matrix cores at float32 accuracy: the activations are
// three bf16 planes (mllm_planes.h, exact), the weights one, two or three
// (gp_planes), and the products above 2^-26 of the largest are formed:
// x0 w0, x1 w0, x2 w0 (1 plane), + x0 w1, x1 w1 (2), + x0 w2 (3).  x0 w0 has an
// accumulator of its own, the corrections share another, added at the end, so
// the roundings of the large sum are one per 16 columns.
//
// No kernel needs a whole row except the norms' statistics, so nothing but the
// GEMMs and the attention is launched for a llama layer:
//   QKV    y = r_t (W (x g)): planes of x g from the kernel that formed x,
//          r_t = 1 / sqrt(mean x^2 + eps) from that kernel's per-64-column
//          sums; epilogue RoPE, q, K and V to the cache
//   ATTN   mllm_prefill.hip's attention, its output written as planes
//   O      x += W_o o; planes of x g2 and the sums of squares of x
//   UP     gate and up rows of the same units: silu(g) u as planes
//   DOWN   x += W_2 h; planes of x g1' (the next layer's norm) and the sums
// GPT-2's LayerNorm subtracts a mean first, which would cancel in the scaled
// form, so its rows are normalised by a kernel of their own.
//
// What bounds it: at a few hundred tokens a launch has fewer wave tiles than
// the chip has SIMDs, and its time is the latency of its loads.  A wave tile is
// 64 rows x 32 tokens; a workgroup is 1 to 8 waves that take slices of the
// columns (added in order through LDS), so that about 1024 waves share the
// loads of a launch.
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
#include "mllm_prefill.h"

namespace mllm {
namespace {

typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

enum { GP_QKV = 0, GP_RESID = 1, GP_SWIGLU = 2, GP_GELU = 3 };
constexpr int GPHD = 64;
constexpr int GPW = 8;               // waves (column slices) of a GEMM workgroup at most
constexpr int GPT = 32 * 68;         // floats of one slice's tile in LDS: 32 tokens x 64 rows (+ 4)
constexpr int GPAD = 3;              // groups read past the end of an operand (never used)

struct GpGemm {
  const uint8_t *w0, *w1;   // tiled rows of sub-tile 0 and 1 (32 rows each)
  const float *s0, *s1;     // per-row scales, or null
  int off1;                 // row tile of sub-tile 1 minus that of sub-tile 0
  int rstep;                // row tiles of the matrix per workgroup (2; 1 where w1 is another matrix)
  int ng;                   // groups per row
  int n, tt0, li, pos0;     // tokens, first token tile, layer, first position
  const uint8_t *px;        // the input's planes
  uint8_t *po;              // the output's planes, or null
  int ldp;                  // groups per token of po
  const float *bias;        // per row, or null
  const float *gain;        // RESID: the next norm's gains (po = planes of x gain), or null
  int rms;                  // the input is x g: scale by 1 / sqrt(mean x^2 + eps)
};

template <int NP>
struct GpLd {
  v8b x[3][2], w[2][NP][2];
};

__device__ __forceinline__ v8b ld_op(const uint8_t *p) {
  return __builtin_bit_cast(v8b, *reinterpret_cast<const uint4 *>(p));
}

__device__ __forceinline__ v16f mfma(v8b a, v8b b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// One group of one sub-tile: hi += w0 x0, lo += the corrections.
template <int NP>
__device__ __forceinline__ void gp_group(const v8b (&x)[3][2], const v8b (&w)[NP][2], v16f &hi, v16f &lo) {
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    hi = mfma(w[0][m], x[0][m], hi);
    lo = mfma(w[0][m], x[1][m], lo);
    lo = mfma(w[0][m], x[2][m], lo);
    if constexpr (NP > 1) {
      lo = mfma(w[1][m], x[0][m], lo);
      lo = mfma(w[1][m], x[1][m], lo);
    }
    if constexpr (NP > 2) lo = mfma(w[2][m], x[0][m], lo);
  }
}

// Dynamic LDS: blockDim / 64 tiles of GPT floats, then 32 floats.
template <int EPI, int NP>
__global__ __launch_bounds__(64 * GPW) void k_gp_gemm(GpArgs A, GpGemm G) {
  extern __shared__ __attribute__((aligned(16))) float buf[];
  const int KS = blockDim.x >> 6, ks = tid() >> 6, lane = tid() & 63, j = lane & 31, hh = lane >> 5;
  // the workgroups of one token tile on one XCD, as in mllm_prefill.hip
  int bx = blockIdx.x, by = blockIdx.y;
  if (gridDim.y % 8 == 0) {
    const int b = bx + (int)gridDim.x * by, k = b >> 3;
    by = (b & 7) + 8 * (k / (int)gridDim.x);
    bx = k % (int)gridDim.x;
  }
  const int T0 = (G.tt0 + by) * 32, rt = bx * G.rstep;
  const int ng = G.ng, gb = ng * ks / KS, ge = ng * (ks + 1) / KS;
  const uint8_t *wa = G.w0 + (size_t)rt * ng * NP * 2048 + 16 * lane;
  const uint8_t *wb = G.w1 + (size_t)(rt + G.off1) * ng * NP * 2048 + 16 * lane;
  const uint8_t *xa = G.px + (size_t)(G.tt0 + by) * ng * BPX + 16 * lane;
  auto load = [&](int g) {
    GpLd<NP> L;
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int m = 0; m < 2; ++m) L.x[p][m] = ld_op(xa + (size_t)g * BPX + (2 * p + m) * 1024);
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        L.w[0][p][m] = ld_op(wa + ((size_t)g * NP + p) * 2048 + m * 1024);
        L.w[1][p][m] = ld_op(wb + ((size_t)g * NP + p) * 2048 + m * 1024);
      }
    return L;
  };
  constexpr int RD = NP == 1 ? 3 : 2;  // groups of loads in flight (the registers they take)
  static_assert(RD <= GPAD, "operands are padded for the read-ahead");
  GpLd<NP> ring[RD];
#pragma unroll
  for (int i = 0; i < RD; ++i) ring[i] = load(gb + i);
  float *rs = buf + KS * GPT;
  if (G.rms && tid() < 32) {  // the tokens' norm scales
    const int nb = A.D >> 6;
    const float *sp = A.ss + (size_t)(T0 + tid()) * nb;
    float s = 0.f;
    for (int b = 0; b < nb; ++b) s += sp[b];
    rs[tid()] = 1.0f / sqrtf(s / (float)A.D + A.eps);
  }
  v16f h0, h1, l0, l1;
#pragma unroll
  for (int v = 0; v < 16; ++v) h0[v] = h1[v] = l0[v] = l1[v] = 0.f;
  for (int g0 = gb; g0 < ge; g0 += RD)
#pragma unroll
    for (int i = 0; i < RD; ++i) {
      if (g0 + i >= ge) break;
      const GpLd<NP> cur = ring[i];
      ring[i] = load(g0 + i + RD);
      gp_group<NP>(cur.x, cur.w[0], h0, l0);
      gp_group<NP>(cur.x, cur.w[1], h1, l1);
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
      float4 s = *reinterpret_cast<const float4 *>(p);
      for (int k = 1; k < KS; ++k) {
        const float4 o = *reinterpret_cast<const float4 *>(p + k * GPT);
        s = make_float4(s.x + o.x, s.y + o.y, s.z + o.z, s.w + o.w);
      }
      *reinterpret_cast<float4 *>(p) = s;
    }
    __syncthreads();
  }
  // epilogue: item = (token jt, rows 8c .. 8c+7 of the tile)
  constexpr int CH = EPI == GP_SWIGLU ? 4 : 8;
  for (int it = tid(); it < 32 * CH; it += blockDim.x) {
    const int jt = it / CH, c = it % CH, t = T0 + jt;
    const bool in = t < G.n;
    const float *row = buf + jt * 68;
    const float r = G.rms ? rs[jt] : 1.f;
    if (EPI == GP_QKV) {
      if (!in) continue;
      const int head = rt >> 1, pos = G.pos0 + t;
      const bool is_q = head < A.NH, is_k = !is_q && head < A.NH + A.NKV;
      const int rd = A.rope_dim, half = rd >> 1;
      const bool rope = A.arch == 0 && (is_q || is_k);
      auto at = [&](int d) {
        const float v = row[d] * r;
        return G.s0 ? v * G.s0[head * GPHD + d] : v;
      };
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int d = 8 * c + e;
        float v = at(d);
        if (G.bias) v += G.bias[head * GPHD + d];
        if (rope && d < rd) {
          const float cs = A.rope_cos[(size_t)pos * rd + d], sn = A.rope_sin[(size_t)pos * rd + d];
          v = __builtin_fmaf(v, cs, (d < half ? -at(d + half) : at(d - half)) * sn);
        }
        y[e] = v;
      }
      if (is_q) {
        float4 *o = reinterpret_cast<float4 *>(A.q + (size_t)t * A.D + head * GPHD + 8 * c);
        o[0] = make_float4(y[0], y[1], y[2], y[3]);
        o[1] = make_float4(y[4], y[5], y[6], y[7]);
      } else {
        const int kvh = is_k ? head - A.NH : head - A.NH - A.NKV;
        const size_t k = ((((size_t)G.li * 2 + (is_k ? 0 : 1)) * A.NKV + kvh) * A.max_seq + pos) * GPHD + 8 * c;
        if (A.kv_fp16) {
          uint32_t w[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            w[e] = (uint32_t)__half_as_ushort(__float2half_rn(y[2 * e])) |
                   (uint32_t)__half_as_ushort(__float2half_rn(y[2 * e + 1])) << 16;
          *reinterpret_cast<uint4 *>(reinterpret_cast<__half *>(A.kv) + k) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
          float4 *o = reinterpret_cast<float4 *>(reinterpret_cast<float *>(A.kv) + k);
          o[0] = make_float4(y[0], y[1], y[2], y[3]);
          o[1] = make_float4(y[4], y[5], y[6], y[7]);
        }
      }
    } else if (EPI == GP_RESID) {
      const int d0 = 32 * rt + 8 * c;
      float4 *xp = reinterpret_cast<float4 *>(A.x + (size_t)min(t, G.n - 1) * A.D + d0);
      const float4 xa4 = xp[0], xb4 = xp[1];
      float y[8] = {xa4.x, xa4.y, xa4.z, xa4.w, xb4.x, xb4.y, xb4.z, xb4.w}, sq = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = row[8 * c + e];
        if (G.s0) v *= G.s0[d0 + e];
        if (G.bias) v += G.bias[d0 + e];
        y[e] += v;
        sq += y[e] * y[e];
      }
      sq = sum8f(sq);  // the token's 64 columns of this tile
      if (!in) continue;
      xp[0] = make_float4(y[0], y[1], y[2], y[3]);
      xp[1] = make_float4(y[4], y[5], y[6], y[7]);
      if (G.gain) {
        if (c == 0) A.ss[(size_t)t * (A.D >> 6) + (rt >> 1)] = sq;
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] *= G.gain[d0 + e];
        planes_store8(G.po + ((size_t)(T0 >> 5) * G.ldp + rt) * BPX, jt, c, y);
      }
    } else if (EPI == GP_SWIGLU) {
      if (!in) continue;
      const int u0 = 32 * rt + 8 * c;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float a = row[8 * c + e] * r, b = row[32 + 8 * c + e] * r;
        if (G.s0) a *= G.s0[u0 + e];
        if (G.s1) b *= G.s1[u0 + e];
        y[e] = (a / (1.0f + expf(-a))) * b;  // infer.js:175-181
      }
      planes_store8(G.po + ((size_t)(T0 >> 5) * G.ldp + rt) * BPX, jt, c, y);
    } else {
      if (!in) continue;
      const int u0 = 32 * rt + 8 * c;
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = row[8 * c + e];
        if (G.s0) v *= G.s0[u0 + e];
        if (G.bias) v += G.bias[u0 + e];
        y[e] = 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));  // infer.js:166-172
      }
      planes_store8(G.po + ((size_t)(T0 >> 5) * G.ldp + rt) * BPX, jt, c, y);
    }
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
      planes_store8(A.pxa + (size_t)(t >> 5) * (D >> 5) * BPX, t & 31, c, v);
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
    planes_store8(A.pxa + (size_t)(t >> 5) * (D >> 5) * BPX, t & 31, c, v);
  }
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
    uint32_t p[3][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) bf16_split3(v[e] * sc, p[0][e], p[1][e], p[2][e]);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (k < np)
        *reinterpret_cast<uint4 *>(dst + (tg * np + k) * 2048 + 16 * l) =
            make_uint4(p[k][0] | p[k][1] << 16, p[k][2] | p[k][3] << 16, p[k][4] | p[k][5] << 16, p[k][6] | p[k][7] << 16);
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
size_t gp_lds(int ks) { return sizeof(float) * ((size_t)ks * GPT + 32); }

// Column slices per tile: doubled while the launch has fewer than 1024 waves
// and every slice keeps two groups.
void launch_gemm(int epi, const GpArgs &A, const GpMat &W, GpGemm G, hipStream_t s) {
  const int tiles = W.rows / (32 * G.rstep), tt = (G.n + 31) / 32 - G.tt0;
  int ks = 1;
  while (ks < GPW && tiles * tt * ks < 1024 && G.ng / (2 * ks) >= 2) ks *= 2;
  hipLaunchKernelGGL(kGpKernels[epi][W.np - 1], dim3(tiles, tt), dim3(64 * ks), gp_lds(ks), s, A, G);
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
  return (size_t)(rows >> 5) * (cols >> 5) * np * 2048 + (size_t)GPAD * np * 2048;
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
size_t px_bytes(int tc, int cols) { return al256(((size_t)((tc + 31) / 32) * (cols >> 5) + GPAD) * BPX); }
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
  return 0;
}

int gp_layers(const GpArgs &A, const int32_t *ids, int n, int pos0, bool last, const float **row, hipStream_t s) {
  MLLM_CHECK(n > 0 && n <= A.tc && pos0 >= 0 && pos0 + n <= A.max_seq, "prompt chunk of %d tokens at %d out of range", n,
             pos0);
  MLLM_HIP(hipMemcpyAsync(A.ids, ids, sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
  const bool gpt2 = A.arch == 1;
  const int ntt = (n + 31) / 32, ngd = A.D >> 5;
  hipLaunchKernelGGL(k_gp_embed, dim3(n), dim3(WG), 0, s, A, gpt2 ? nullptr : A.layers[0].n1, pos0);
  PfArgs P{};
  P.D = A.D;
  P.NH = A.NH;
  P.NKV = A.NKV;
  P.max_seq = A.max_seq;
  P.kv_fp16 = A.kv_fp16;
  P.attn_scale = A.attn_scale;
  P.kv = A.kv;
  P.q = A.q;
  P.opx = A.pxo;
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
    pf_attention(P, li, n, pos0, tt0, s);
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
