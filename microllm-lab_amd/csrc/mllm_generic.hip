// mllm_generic.hip -- the decode step for models whose matrices are not all
// Q4 group-32 (infer.js:313-346 binds each matrix by its own storage; the
// reference's GPU engine packs Q8, f16 and bf16 models as they are,
// webgpu.js:902-973, and runs them through the same step with a per-kind
// weight load, webgpu.js:141-260).
//
// One token per step, a few kernels per layer:
//   k_g_embed    the token's row of the tied lm_head in its storage
//                (infer.js:360-420: quantised rows de-scaled by gpt2's
//                scale_factors) + gpt2's learned position
//   k_g_gemv     a weight row per segment of lanes, its input row -- with
//                the norm (RMSNorm / LayerNorm) or, for O, the merge of the
//                attention's splits -- in registers; epilogue: store (+ bias),
//                residual add (+ bias), SwiGLU over the w1 / w3 rows, or bias
//                + GELU-tanh
//   k_g_attn     a workgroup per query head and 256 positions: rotate-half
//                RoPE of its q and of its KV group's new k (infer.js:208-225);
//                the group's first head writes k / v to the KV cache (the
//                engine's layout); scores, softmax statistics
//                (infer.js:227-238) and P.V (infer.js:466-495) of its
//                positions
//   k_g_argmax   first maximum (infer.js:240-250), or argmaxGpt2
//                (infer.js:252-287) in gpt2 chains
// These matrices are read once per token, as by the Q4 engine, at the
// bytes their storage takes (f32 4, f16 / bf16 2, Q8 1 per weight).  A
// step's position and token come from a device cursor (GCursor) that the
// step's first kernel advances, so the host replays one captured graph per
// token.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "mllm_device.h"
#include "mllm_generic.h"
#include "mllm_host.h"
#include "mllm_kinds.h"

namespace mllm {
namespace {

constexpr int GHD = 64;   // head dimension
constexpr int GT = 256;   // threads per workgroup
constexpr int GAT = 1024;  // threads of the argmax workgroup
enum { G_STORE = 0, G_RESID = 1, G_SWIGLU = 2, G_GELU = 3 };
enum { GN_NONE = 0, GN_RMS = 1, GN_LN = 2, GN_SPLITS = 3 };
constexpr int GSPLIT = kGenericSplit;  // positions per attention workgroup
constexpr int GAW = 8, GAK = GSPLIT / GAW;  // its waves, the positions of each
constexpr int GAPS = kGenericPart;     // floats of its partial: max, sum, 2 pad, 64 outputs

// Chained calls stop once an EOS was emitted.
__device__ __forceinline__ bool stopped(const GCursor *c) {
  return c && *reinterpret_cast<const volatile int *>(&c->done) != 0;
}

// ---------------------------------------------------------------- GEMV
// A row of the matrix is on a segment of L lanes (a power of two): lane l
// takes the 8-column chunks l, l + L, ... (at most CB of them where L = 64
// allows it), keeps their inputs in registers and dots them in order; a DPP /
// swizzle tree over the segment ends the row.  L follows from the column count
// and the storage alone, so a row's bits do not depend on the launch.
//
// Every segment reads the whole input row, so the RMS norm's mean square and
// the LayerNorm's moments are the same tree: no LDS and no barrier, and every
// load of the kernel -- weights, inputs, gains, what the epilogue needs -- is
// on its way at once.  These launches are bound by that one latency (a layer's
// matrices are 0.2 to 3 MB), where the former form (inputs staged in LDS, two
// to three block reductions, then the weights) paid it two to three times:
// per-row Q8 at the 135M shape, us a launch, QKV 5.1 -> 4.2, O 5.1 -> 4.1 (it
// merges the attention's splits, too), gate/up 6.3 -> 4.9, down 5.1 -> 3.8,
// lm_head 21 -> 12.3.
constexpr int G_MIXED = -1;  // W and W3 of different storages
template <int KIND>
__host__ __device__ constexpr int g_cb() {
  return KIND == MLLM_F32 || KIND == G_MIXED ? 4 : 8;
}

// A chunk as loaded and its scale.
template <int KIND>
struct Raw {
  uint32_t d[KIND == MLLM_F32 || KIND == G_MIXED ? 8 : KIND == MLLM_F16 || KIND == MLLM_BF16 ? 4 : KIND == MLLM_Q4 ? 1 : 2];
  float sc;
};

template <int KIND>
__device__ __forceinline__ Raw<KIND> raw_load(const GMat &W, int r, int c) {
  Raw<KIND> R;
  R.sc = 1.f;
  if constexpr (KIND == G_MIXED) {
    float w[8];
    R.sc = load8(W, r, c, w);
#pragma unroll
    for (int e = 0; e < 8; ++e) R.d[e] = __float_as_uint(w[e]);
  } else {
    const size_t e0 = (size_t)r * W.cols + 8 * (size_t)c;
    const uint8_t *p = static_cast<const uint8_t *>(W.w);
    if constexpr (KIND == MLLM_F32) {
      const uint4 a = *reinterpret_cast<const uint4 *>(p + 4 * e0), b = *reinterpret_cast<const uint4 *>(p + 4 * e0 + 16);
      R.d[0] = a.x, R.d[1] = a.y, R.d[2] = a.z, R.d[3] = a.w, R.d[4] = b.x, R.d[5] = b.y, R.d[6] = b.z, R.d[7] = b.w;
    } else if constexpr (KIND == MLLM_F16 || KIND == MLLM_BF16) {
      const uint4 a = *reinterpret_cast<const uint4 *>(p + 2 * e0);
      R.d[0] = a.x, R.d[1] = a.y, R.d[2] = a.z, R.d[3] = a.w;
    } else if constexpr (KIND == MLLM_Q4) {
      R.d[0] = *reinterpret_cast<const uint32_t *>(p + e0 / 2);
      R.sc = W.s[(size_t)r * (W.cols / W.group) + (8 * c) / W.group];
    } else {
      const uint2 a = *reinterpret_cast<const uint2 *>(p + e0);
      R.d[0] = a.x, R.d[1] = a.y;
      if (KIND == MLLM_Q8G32) R.sc = W.s[(size_t)r * (W.cols >> 5) + (c >> 2)];
    }
  }
  return R;
}

template <int KIND>
__device__ __forceinline__ float raw_at(const Raw<KIND> &R, int e) {
  if constexpr (KIND == MLLM_F32 || KIND == G_MIXED) return __uint_as_float(R.d[e]);
  if constexpr (KIND == MLLM_F16) return f16_bits(e & 1 ? R.d[e >> 1] >> 16 : R.d[e >> 1] & 0xffffu);
  if constexpr (KIND == MLLM_BF16) return __uint_as_float(e & 1 ? R.d[e >> 1] & 0xffff0000u : R.d[e >> 1] << 16);
  if constexpr (KIND == MLLM_Q4) return (float)((int)((R.d[0] >> (4 * e)) & 15u) - 8);  // byte k: elements 2k, 2k + 1
  return (float)(int8_t)(R.d[e >> 2] >> (8 * (e & 3)));
}

template <int KIND>
__device__ __forceinline__ float raw_dot(const Raw<KIND> &R, const float (&x)[8], float acc) {
  float d = raw_at<KIND>(R, 0) * x[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) d = __builtin_fmaf(raw_at<KIND>(R, e), x[e], d);
  if constexpr (KIND == MLLM_Q4 || KIND == MLLM_Q8G32 || KIND == G_MIXED) return __builtin_fmaf(d, R.sc, acc);
  return acc + d;
}

struct GemvArgs {
  GMat W, W3;          // W3: the up rows of G_SWIGLU
  const float *x;      // input row [W.cols] (GN_SPLITS: the attention's partials)
  const float *gains;  // norm gains (LayerNorm: gamma || beta) or null
  float eps;           // RMSNorm eps (LayerNorm: 1e-5, infer.js:145)
  const float *bias;   // per output row, or null
  float *y;            // output row [W.rows]; G_RESID adds to it
  int L;               // lanes per row
  int rp;              // row groups (64 / L rows) per wave
  const GCursor *cur;
  int lm;              // 1: y is the logits, row cur->i when cur->rows (verify)
  int nsplit_max;      // GN_SPLITS: partials per head in x
  int m, xs;           // tokens of the pass and the stride of their inputs (outputs: W.rows)
};

// The attention's output row from its splits' partials (infer.js:466-495) into
// LDS: a thread per four components, its splits' loads four at a time.
__device__ __forceinline__ void merge_splits(const GemvArgs &a, int tok, float *sx) {
  const int ns = (a.cur->pos + tok) / GSPLIT + 1;
  for (int i = tid(); i < (a.W.cols >> 2); i += GT) {
    const float *p = a.x + (size_t)tok * a.xs + (size_t)(i >> 4) * a.nsplit_max * GAPS;
    float mx = -INFINITY, l = 0.f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = 0; s0 < ns; s0 += 4) {
      float m[4], ls[4];
      float4 u[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float *q = p + min(s0 + k, ns - 1) * GAPS;
        const float2 ml = *reinterpret_cast<const float2 *>(q);
        m[k] = s0 + k < ns ? ml.x : -INFINITY;
        ls[k] = ml.y;
        u[k] = *reinterpret_cast<const float4 *>(q + 4 + 4 * (i & 15));
      }
      const float mn = fmaxf(mx, fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3])));
      const float ref = score_ref(mn), f0 = expf(mx - ref);  // 0 at first
      l *= f0, o.x *= f0, o.y *= f0, o.z *= f0, o.w *= f0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float f = expf(m[k] - ref);
        l = __builtin_fmaf(ls[k], f, l);
        o.x = __builtin_fmaf(u[k].x, f, o.x), o.y = __builtin_fmaf(u[k].y, f, o.y);
        o.z = __builtin_fmaf(u[k].z, f, o.z), o.w = __builtin_fmaf(u[k].w, f, o.w);
      }
      mx = mn;
    }
    const float inv = 1.0f / l;
    *reinterpret_cast<float4 *>(sx + 4 * i) = make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv);
  }
}

__device__ __forceinline__ void vec8(const float *p, int c, float (&v)[8]) {
  const float4 u0 = ld4u(p + 8 * c), u1 = ld4u(p + 8 * c + 4);
  v[0] = u0.x, v[1] = u0.y, v[2] = u0.z, v[3] = u0.w, v[4] = u1.x, v[5] = u1.y, v[6] = u1.z, v[7] = u1.w;
}

__device__ __forceinline__ void in8(const float *x, int c, float (&v)[8]) {  // 16-byte aligned
  const float4 u0 = *reinterpret_cast<const float4 *>(x + 8 * c), u1 = *reinterpret_cast<const float4 *>(x + 8 * c + 4);
  v[0] = u0.x, v[1] = u0.y, v[2] = u0.z, v[3] = u0.w, v[4] = u1.x, v[5] = u1.y, v[6] = u1.z, v[7] = u1.w;
}

// What a row's end reads besides the sums, loaded with the weights.
struct RowEnd {
  float s, s3, bias, y;
};
template <int EPI>
__device__ __forceinline__ RowEnd row_end(const GemvArgs &a, const float *y, int r) {
  RowEnd E{1.f, 1.f, 0.f, 0.f};
  if (a.W.kind == MLLM_Q8) E.s = a.W.s[r];
  if (EPI == G_SWIGLU && a.W3.kind == MLLM_Q8) E.s3 = a.W3.s[r];
  if (EPI != G_SWIGLU && a.bias) E.bias = a.bias[r];
  if (EPI == G_RESID) E.y = y[r];
  return E;
}
template <int EPI>
__device__ __forceinline__ float row_out(const GemvArgs &a, const RowEnd &E, float acc, float acc3) {
  if (a.W.kind == MLLM_Q8) acc *= E.s;
  if (EPI == G_SWIGLU) {
    if (a.W3.kind == MLLM_Q8) acc3 *= E.s3;
    return (acc / (1.0f + expf(-acc))) * acc3;  // infer.js:175-181
  }
  if (a.bias) acc += E.bias;
  if (EPI == G_RESID) return E.y + acc;
  if (EPI == G_GELU) return 0.5f * acc * (1.0f + tanhf(0.7978845608028654f * (acc + 0.044715f * acc * acc * acc)));  // infer.js:166-172
  return acc;
}

// Loads above are issued before what is below: without it the compiler moves
// the weights' loads under the branches that follow.
__device__ __forceinline__ void loads_first() { asm volatile("" ::: "memory"); }

// GN_SPLITS: W.cols floats of dynamic LDS.
template <int KIND, int EPI, int NORM>
__global__ __launch_bounds__(GT) void k_g_gemv(GemvArgs a) {
  extern __shared__ __attribute__((aligned(16))) float sx[];
  constexpr int CB = g_cb<KIND>();
  const int K = a.W.cols, nc = K >> 3, L = a.L, nch = (nc + L - 1) / L, rows = a.W.rows;
  const int lane = tid() & 63, l = lane & (L - 1), seg = lane / L, rpw = 64 / L;
  const int g0 = ((int)blockIdx.x * (GT / 64) + (tid() >> 6)) * a.rp;
  auto chunk = [&](int k) { return min(l + k * L, nc - 1); };  // past the row: a valid chunk, its input taken as 0
  auto row_of = [&](int g) { return min(g * rpw + seg, rows - 1); };
  const GCursor *cur = a.cur;
  const int tok = blockIdx.y;  // passes of several tokens: a weight row's workgroups meet it in the caches
  if (nch <= CB) {
    // every load of the first rows and of the input row, then the rest
    Raw<KIND> w[CB], w3[EPI == G_SWIGLU ? CB : 1];
    auto load = [&](int g) {
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) {
          w[k] = raw_load<KIND>(a.W, row_of(g), chunk(k));
          if (EPI == G_SWIGLU) w3[k] = raw_load<KIND>(a.W3, row_of(g), chunk(k));
        }
    };
    float x[CB][8], gv[NORM == GN_RMS || NORM == GN_LN ? CB : 1][8], scale = 1.f;
    if (NORM != GN_SPLITS) {
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) in8(a.x + (size_t)tok * a.xs, chunk(k), x[k]);
    }
    load(g0);
    if (NORM == GN_RMS || NORM == GN_LN) {
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) vec8(a.gains, chunk(k), gv[k]);
    }
    float *y = a.y + (size_t)tok * rows;
    RowEnd E = row_end<EPI>(a, y, row_of(g0));
    loads_first();
    if (cur) {
      if (stopped(cur)) return;
      if (a.lm && cur->rows) y += (size_t)cur->i * rows;
    }
    if (NORM == GN_SPLITS) {
      merge_splits(a, tok, sx);
      __syncthreads();
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) in8(sx, chunk(k), x[k]);
    }
    if (g0 * rpw >= rows) return;  // uniform in the wave
    if (NORM == GN_RMS) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) {
          float s = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            s = __builtin_fmaf(x[k][e], x[k][e], s);
            x[k][e] *= gv[k][e];
          }
          ss += l + k * L < nc ? s : 0.f;
        }
      scale = 1.0f / sqrtf(seg_sum(ss, L) / (float)K + a.eps);
    } else if (NORM == GN_LN) {
      float bv[CB][8], s = 0.f;
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) vec8(a.gains + K, chunk(k), bv[k]);
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) {
          float t = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) t += x[k][e];
          s += l + k * L < nc ? t : 0.f;
        }
      const float mean = seg_sum(s, L) / (float)K;
      s = 0.f;
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) {
          float t = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            x[k][e] -= mean;
            t = __builtin_fmaf(x[k][e], x[k][e], t);
          }
          s += l + k * L < nc ? t : 0.f;
        }
      const float r = 1.0f / sqrtf(seg_sum(s, L) / (float)K + 1e-5f);
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[k][e] = __builtin_fmaf(x[k][e] * r, gv[k][e], bv[k][e]);
        }
    }
#pragma unroll
    for (int k = 0; k < CB; ++k)
      if (k < nch && l + k * L >= nc) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[k][e] = 0.f;
      }
    for (int i = 0; i < a.rp; ++i) {
      const int g = g0 + i;
      if (g * rpw >= rows) break;
      float acc = 0.f, acc3 = 0.f;
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k < nch) {
          acc = raw_dot<KIND>(w[k], x[k], acc);
          if (EPI == G_SWIGLU) acc3 = raw_dot<KIND>(w3[k], x[k], acc3);
        }
      const RowEnd E0 = E;
      if (i + 1 < a.rp) {  // the next rows' weights while this sum ends
        load(g + 1);
        E = row_end<EPI>(a, y, row_of(g + 1));
      }
      acc = seg_sum(acc, L) * scale;
      if (EPI == G_SWIGLU) acc3 = seg_sum(acc3, L) * scale;
      const int r = g * rpw + seg;
      const float o = row_out<EPI>(a, E0, acc, acc3);
      if (l == 0 && r < rows) y[r] = o;
    }
    return;
  }
  // rows past the registers (L = 64): the moments first, then CB chunks at a time
  if (cur && stopped(cur)) return;
  float *y = a.y + (a.lm && cur->rows ? (size_t)cur->i * rows : 0) + (size_t)tok * rows;
  if (NORM == GN_SPLITS) {
    merge_splits(a, tok, sx);
    __syncthreads();
  }
  const float *x = NORM == GN_SPLITS ? sx : a.x + (size_t)tok * a.xs;
  float scale = 1.f, mean = 0.f;
  if (NORM == GN_RMS || NORM == GN_LN) {
    float s = 0.f;
    for (int k = 0; k < nch; ++k) {
      float v[8], t = 0.f;
      in8(x, chunk(k), v);
#pragma unroll
      for (int e = 0; e < 8; ++e) t = NORM == GN_RMS ? __builtin_fmaf(v[e], v[e], t) : t + v[e];
      s += l + k * L < nc ? t : 0.f;
    }
    s = seg_sum(s, L) / (float)K;
    if (NORM == GN_RMS) {
      scale = 1.0f / sqrtf(s + a.eps);
    } else {
      mean = s;
      s = 0.f;
      for (int k = 0; k < nch; ++k) {
        float v[8], t = 0.f;
        in8(x, chunk(k), v);
#pragma unroll
        for (int e = 0; e < 8; ++e) t = __builtin_fmaf(v[e] - mean, v[e] - mean, t);
        s += l + k * L < nc ? t : 0.f;
      }
      scale = 1.0f / sqrtf(seg_sum(s, L) / (float)K + 1e-5f);
    }
  }
  for (int i = 0; i < a.rp && (g0 + i) * rpw < rows; ++i) {
    const int r = row_of(g0 + i);
    const RowEnd E = row_end<EPI>(a, y, r);
    float acc = 0.f, acc3 = 0.f;
    for (int k0 = 0; k0 < nch; k0 += CB)
#pragma unroll
      for (int k = 0; k < CB; ++k)
        if (k0 + k < nch) {
          const int c = chunk(k0 + k);
          const Raw<KIND> w = raw_load<KIND>(a.W, r, c);
          float v[8];
          in8(x, c, v);
          if (NORM == GN_RMS || NORM == GN_LN) {
            float gv[8], bv[8];
            vec8(a.gains, c, gv);
            if (NORM == GN_LN) vec8(a.gains + K, c, bv);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              v[e] = NORM == GN_LN ? __builtin_fmaf((v[e] - mean) * scale, gv[e], bv[e]) : v[e] * scale * gv[e];
          }
          if (l + (k0 + k) * L >= nc) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = 0.f;
          }
          acc = raw_dot<KIND>(w, v, acc);
          if (EPI == G_SWIGLU) acc3 = raw_dot<KIND>(raw_load<KIND>(a.W3, r, c), v, acc3);
        }
    acc = seg_sum(acc, L);
    if (EPI == G_SWIGLU) acc3 = seg_sum(acc3, L);
    const float o = row_out<EPI>(a, E, acc, acc3);
    if (l == 0 && (g0 + i) * rpw + seg < rows) y[r] = o;
  }
}

__device__ __forceinline__ size_t g_kv_index(const GArgs &A, int li, int which, int h, int pos) {
  return ((((size_t)li * 2 + which) * A.NKV + h) * A.max_seq + pos) * GHD;
}

// The step's start: position and token index from the cursor (advanced for
// the next step), the input token (chained calls: the previous argmax),
// its embedding row.
__global__ __launch_bounds__(GT) void k_g_embed(GArgs A) {
  GCursor *cur = A.cur;
  if (stopped(cur)) return;
  // a pass of several tokens (a workgroup each) starts from a cursor that the
  // host has set and leaves it alone
  const bool pass = gridDim.x > 1;
  const int D = A.D, pos = pass ? cur->pos + (int)blockIdx.x : cur->pos_next, ti = pass ? (int)blockIdx.x : cur->i_next;
  const int id = cur->chain ? cur->tok : A.ids[ti];
  float *x = A.x + (size_t)blockIdx.x * D;
  __syncthreads();  // every thread has read the cursor
  if (tid() == 0 && !pass) {
    cur->pos = pos;
    cur->i = ti;
    cur->pos_next = pos + 1;
    cur->i_next = ti + 1;
  }
  const GMat &W = A.lm;
  const bool quant = W.kind == MLLM_Q8 || W.kind == MLLM_Q8G32 || W.kind == MLLM_Q4;
  for (int c = tid(); c < (D >> 3); c += GT) {
    float w[8];
    const float sc = load8(W, id, c, w);
    const float rs = W.kind == MLLM_Q8 ? W.s[id] : sc;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = 8 * c + e;
      float v = quant ? w[e] * rs : w[e];
      if (A.arch == 1) {
        if (quant && A.sf) v = v / A.sf[i];
        v = v + A.wpe[(size_t)min(pos, A.max_seq - 1) * D + i];
      }
      x[i] = v;
    }
  }
}

// One head's rotated component d (rotate-half on the first rope_dim
// components: out[d] = x[d] cos[d] + rot[d] sin[d], rot = (-x[half .. rd),
// x[0 .. half))).
__device__ __forceinline__ float rope_at(const GArgs &A, const float *hd, int d, int pos) {
  const int rd = A.rope_dim, half = rd >> 1;
  if (A.arch != 0 || d >= rd) return hd[d];
  const float c = A.rope_cos[(size_t)pos * rd + d], sn = A.rope_sin[(size_t)pos * rd + d];
  return d < half ? hd[d] * c + (-hd[d + half]) * sn : hd[d] * c + hd[d - half] * sn;
}

// Workgroup (query head h, 256 positions), wave w on 32 of them: 16 lanes hold
// a cached row (4 components each), so a load instruction of the wave reads
// four rows, 1 KiB in f32, and all 16 of a wave go out before its first score.
// Each wave forms its scores, their softmax statistics and P.V by itself; the
// workgroup's eight are merged in wave order (max, sum of weights, outputs) into
// attp, and the O GEMV merges the splits while it reads its input.  The
// former form -- a workgroup per head, a row per thread, then P.V down four
// position slices -- was bound by one workgroup's load rate: 32.2 us at 700
// positions of the 135M shape, 7.2 now (8.3 with 64 positions a wave: twice
// the code, which runs once from a cold instruction cache).
// The new position's k and v are taken from LDS (as the cache holds them:
// f16-rounded for an f16 cache), so a group's heads do not wait for the one
// that writes them to the cache.
template <bool F16>
__global__ __launch_bounds__(GAW * 64) void k_g_attn(GArgs A, int li) {
  __shared__ __attribute__((aligned(16))) float own[GAW][3 * GHD];  // each wave's q, new k, new v
  __shared__ float part[GAW][GHD + 2];
  const int tok = blockIdx.z;
  const int done = A.cur->done, pos = A.cur->pos + tok, rep = A.NH / A.NKV, n = pos + 1;  // one load
  if (done) return;
  const int h = blockIdx.x, kvh = h / rep, lane = tid() & 63, wv = tid() >> 6;
  const int s0 = (int)blockIdx.y * GSPLIT;
  if (s0 >= n) return;
  constexpr int ES = F16 ? 2 : 4;  // bytes of a cache element
  const size_t kb = g_kv_index(A, li, 0, kvh, 0), vb = g_kv_index(A, li, 1, kvh, 0);
  const int k0 = s0 + GAK * wv;  // this wave's positions k0 .. k0 + GAK - 1
  const bool on = k0 < n;       // uniform in the wave
  // q, k, v rows of the step, one component per lane (these loads first)
  float *qs = own[wv], *kn = qs + GHD, *vn = kn + GHD;
  const float *qkv = A.qkv + (size_t)tok * (A.D + 2 * A.NKV * GHD), *kq = qkv + A.D + kvh * GHD;
  const float qv = rope_at(A, qkv + h * GHD, lane, pos);
  float kv = rope_at(A, kq, lane, pos), vv = kq[A.NKV * GHD + lane];
  const int grp = lane >> 4, d4 = 4 * (lane & 15);
  uint4 kr[GAK / 4], vr[GAK / 4];
  if (on) {
    // resources of the rows before the new one (none at position 0): the row at
    // it, which another head may be writing, and those past it, left by earlier
    // calls, are read as 0 -- their weight is 0, and 0 times an infinity is NaN
    uint8_t *cache = static_cast<uint8_t *>(A.kv);
    const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc(cache + kb * ES, (short)0, pos * GHD * ES, 0x00020000);
    const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc(cache + vb * ES, (short)0, pos * GHD * ES, 0x00020000);
    const int at = ((k0 + grp) * GHD + d4) * ES;
#pragma unroll
    for (int i = 0; i < GAK / 4; ++i) {
      const int off = at + 4 * i * GHD * ES;
      if (F16) {
        const uint2 a = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(kres, off, 0, 0));
        const uint2 b = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(vres, off, 0, 0));
        kr[i] = make_uint4(a.x, a.y, 0u, 0u);
        vr[i] = make_uint4(b.x, b.y, 0u, 0u);
      } else {
        kr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(kres, off, 0, 0));
        vr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(vres, off, 0, 0));
      }
    }
  }
  // (passes of several tokens: k_g_kv has written them)
  const bool writes = gridDim.z == 1 && h % rep == 0 && pos >= k0 && pos < k0 + GAK;  // uniform in the wave
  if (F16) {
    const __half kh = __float2half_rn(kv), vh = __float2half_rn(vv);
    kv = __half2float(kh);
    vv = __half2float(vh);
    if (writes) {
      reinterpret_cast<__half *>(A.kv)[kb + (size_t)pos * GHD + lane] = kh;
      reinterpret_cast<__half *>(A.kv)[vb + (size_t)pos * GHD + lane] = vh;
    }
  } else if (writes) {
    reinterpret_cast<float *>(A.kv)[kb + (size_t)pos * GHD + lane] = kv;
    reinterpret_cast<float *>(A.kv)[vb + (size_t)pos * GHD + lane] = vv;
  }
  qs[lane] = qv;
  kn[lane] = kv;
  vn[lane] = vv;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();  // the wave's own rows, read below by its other lanes
  float m = -INFINITY, sum = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  auto row = [&](const uint4 &u) {
    if (!F16)
      return make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
    return make_float4(f16_bits(u.x & 0xffffu), f16_bits(u.x >> 16), f16_bits(u.y & 0xffffu), f16_bits(u.y >> 16));
  };
  if (on) {
    const float4 q = *reinterpret_cast<const float4 *>(qs + d4), kl = *reinterpret_cast<const float4 *>(kn + d4),
                 vl = *reinterpret_cast<const float4 *>(vn + d4);
    float sc[GAK / 4];
#pragma unroll
    for (int i = 0; i < GAK / 4; ++i) {
      const int key = k0 + 4 * i + grp;
      const float4 k = key == pos ? kl : row(kr[i]);
      const float d = row16_sum(__builtin_fmaf(q.w, k.w, __builtin_fmaf(q.z, k.z, __builtin_fmaf(q.y, k.y, q.x * k.x))));
      sc[i] = key < n ? d * A.attn_scale : -INFINITY;
      m = fmaxf(m, sc[i]);
    }
    m = fmaxf(m, __shfl_xor(m, 16));
    m = fmaxf(m, __shfl_xor(m, 32));
    const float ref = score_ref(m);
#pragma unroll
    for (int i = 0; i < GAK / 4; ++i) {
      const float p = expf(sc[i] - ref);
      const float4 v = k0 + 4 * i + grp == pos ? vl : row(vr[i]);
      sum += p;
      o.x = __builtin_fmaf(p, v.x, o.x);
      o.y = __builtin_fmaf(p, v.y, o.y);
      o.z = __builtin_fmaf(p, v.z, o.z);
      o.w = __builtin_fmaf(p, v.w, o.w);
    }
#pragma unroll
    for (int x = 16; x < 64; x *= 2) {
      sum += __shfl_xor(sum, x);
      o.x += __shfl_xor(o.x, x);
      o.y += __shfl_xor(o.y, x);
      o.z += __shfl_xor(o.z, x);
      o.w += __shfl_xor(o.w, x);
    }
  }
  if (lane < 16) {
    part[wv][d4] = o.x;
    part[wv][d4 + 1] = o.y;
    part[wv][d4 + 2] = o.z;
    part[wv][d4 + 3] = o.w;
    if (lane == 0) {
      part[wv][GHD] = m;
      part[wv][GHD + 1] = sum;
    }
  }
  __syncthreads();
  if (wv != 0) return;
  float mx = part[0][GHD];
#pragma unroll
  for (int w = 1; w < GAW; ++w) mx = fmaxf(mx, part[w][GHD]);
  const float ref = score_ref(mx);
  float l = 0.f, out = 0.f;
#pragma unroll
  for (int w = 0; w < GAW; ++w) {
    const float f = expf(part[w][GHD] - ref);  // 0 for a wave without positions
    l = __builtin_fmaf(part[w][GHD + 1], f, l);
    out = __builtin_fmaf(part[w][lane], f, out);
  }
  float *p = A.attp + (((size_t)tok * A.NH + h) * gridDim.y + blockIdx.y) * GAPS;
  p[4 + lane] = out;
  if (lane == 0) {
    p[0] = mx;
    p[1] = l;
  }
}

// A pass of several tokens: their k and v rows to the cache before the
// attention, whose later tokens read the earlier ones' from there (a
// workgroup's 64 lanes: one KV head of one token).
template <bool F16>
__global__ __launch_bounds__(GHD) void k_g_kv(GArgs A, int li) {
  const int kvh = blockIdx.x, tok = blockIdx.y, pos = A.cur->pos + tok, lane = tid();
  const float *kq = A.qkv + (size_t)tok * (A.D + 2 * A.NKV * GHD) + A.D + kvh * GHD;
  const float kv = rope_at(A, kq, lane, pos), vv = kq[A.NKV * GHD + lane];
  const size_t kb = g_kv_index(A, li, 0, kvh, pos) + lane, vb = g_kv_index(A, li, 1, kvh, pos) + lane;
  if (F16) {
    reinterpret_cast<__half *>(A.kv)[kb] = __float2half_rn(kv);
    reinterpret_cast<__half *>(A.kv)[vb] = __float2half_rn(vv);
  } else {
    reinterpret_cast<float *>(A.kv)[kb] = kv;
    reinterpret_cast<float *>(A.kv)[vb] = vv;
  }
}

// First maximum of the step's logits row (infer.js:240-250: NaN never
// wins, and a NaN in slot 0 keeps index 0); in a gpt2 chain argmaxGpt2
// over the history (infer.js:252-287: trigram-banned ids -1e9, ids among
// the last 32 scaled by 1/1.15 or 1.15, then the first strict maximum from
// -inf).  Dynamic LDS: 2 + 32 + max_seq ints.
__global__ __launch_bounds__(GAT) void k_g_argmax(GArgs A) {
  extern __shared__ int lists[];
  GCursor *cur = A.cur;
  if (stopped(cur)) return;
  const int row = (cur->rows ? cur->i : 0) + (int)blockIdx.x, chained = cur->chain;
  const float *lg = A.logits + (size_t)row * A.V;
  const bool rule = chained && cur->gpt2_rule;
  int *nb = lists, *nr = lists + 1, *rec = lists + 2, *ban = lists + 34;
  const int nh = chained ? cur->n_hist + cur->emitted : 0;
  const int *hist = A.hist;
  if (rule) {
    if (tid() == 0) {
      *nb = 0;
      int k = 0;
      for (int h = max(0, nh - 32); h < nh; ++h) rec[k++] = hist[h];
      *nr = k;
    }
    __syncthreads();
    if (nh >= 2) {
      const int t1 = hist[nh - 2], t2 = hist[nh - 1];
      for (int h = tid(); h < nh - 2; h += GAT)
        if (hist[h] == t1 && hist[h + 1] == t2) ban[atomicAdd(nb, 1)] = hist[h + 2];
    }
    __syncthreads();
  }
  const int nban = rule ? *nb : 0, nrec = rule ? *nr : 0;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  auto take = [&](float v, int i) {
    if (rule) {
      for (int k = 0; k < nban; ++k)
        if (ban[k] == i) {
          v = -1e9f;
          break;
        }
      if (v > -1e8f)
        for (int k = 0; k < nrec; ++k)
          if (rec[k] == i) {
            v = v > 0.f ? v / 1.15f : v * 1.15f;
            break;
          }
    }
    // candidates: values above -inf (NaN and -inf never displace a maximum)
    if (v > -INFINITY && amax_better(v, i, bv, bi)) {
      bv = v;
      bi = i;
    }
  };
  // 32 KiB of loads at a time (one workgroup: its loads in flight bound it;
  // 49152 logits one by one took 19.4 us, 16 KiB at a time 9.5)
  int i0 = 0;
  constexpr int AB = 8;
  for (; i0 + AB * GAT <= A.V; i0 += AB * GAT) {
    float v[AB];
#pragma unroll
    for (int k = 0; k < AB; ++k) v[k] = lg[i0 + k * GAT + tid()];
#pragma unroll
    for (int k = 0; k < AB; ++k) take(v[k], i0 + k * GAT + tid());
  }
  for (int i = i0 + tid(); i < A.V; i += GAT) take(lg[i], i);
  wave_argmax(bv, bi);
  __shared__ float wv_v[GAT / 64];
  __shared__ int wv_i[GAT / 64];
  if ((tid() & 63) == 0) {
    wv_v[tid() >> 6] = bv;
    wv_i[tid() >> 6] = bi;
  }
  __syncthreads();
  if (tid() != 0) return;
  for (int w = 1; w < GAT / 64; ++w)
    if (amax_better(wv_v[w], wv_i[w], bv, bi)) {
      bv = wv_v[w];
      bi = wv_i[w];
    }
  int best = bi == 0x7fffffff ? 0 : bi;  // nothing above -inf: index 0 (both rules)
  if (!rule && isnan(lg[0])) best = 0;   // infer.js:241-243 starts from logits[0]
  A.res[row] = best;
  if (chained) {
    A.hist[nh] = best;
    cur->tok = best;
    cur->emitted = cur->emitted + 1;
    if (best == cur->eos) cur->done = 1;
  }
}

// Lanes per row: the fewest (8 or more, a power of two) that keep a lane's
// chunks in registers -- g_cb, 6 for a LayerNorm's row in 8-chunk storages,
// whose gains and shifts are held beside it -- else all 64.
template <int KIND>
int g_lanes(int cols, bool ln) {
  const int nc = cols / 8, cb = ln ? std::min(6, g_cb<KIND>()) : g_cb<KIND>();
  int L = 8;
  while (L < 64 && (nc + L - 1) / L > cb) L *= 2;
  return L;
}

template <int KIND, int EPI, int NORM>
void launch_kind(GemvArgs a, hipStream_t s) {
  a.L = g_lanes<KIND>(a.W.cols, NORM == GN_LN);
  const int groups = (a.W.rows + 64 / a.L - 1) / (64 / a.L);
  // one row group per wave up to 4096 waves (the input row is read by each
  // wave: beyond that they would read more input than weights)
  a.rp = std::max(1, (groups + 4095) / 4096);
  const int waves = (groups + a.rp - 1) / a.rp;
  hipLaunchKernelGGL((k_g_gemv<KIND, EPI, NORM>), dim3((waves + GT / 64 - 1) / (GT / 64), a.m), dim3(GT),
                     NORM == GN_SPLITS ? sizeof(float) * a.W.cols : 0, s, a);
}

template <int EPI, int NORM>
void launch_gemv(const GemvArgs &a, hipStream_t s) {
  switch (EPI == G_SWIGLU && a.W3.kind != a.W.kind ? G_MIXED : a.W.kind) {
  case MLLM_F32: return launch_kind<MLLM_F32, EPI, NORM>(a, s);
  case MLLM_F16: return launch_kind<MLLM_F16, EPI, NORM>(a, s);
  case MLLM_BF16: return launch_kind<MLLM_BF16, EPI, NORM>(a, s);
  case MLLM_Q8: return launch_kind<MLLM_Q8, EPI, NORM>(a, s);
  case MLLM_Q8G32: return launch_kind<MLLM_Q8G32, EPI, NORM>(a, s);
  case MLLM_Q4: return launch_kind<MLLM_Q4, EPI, NORM>(a, s);
  default: return launch_kind<G_MIXED, EPI, NORM>(a, s);
  }
}

GemvArgs gemv_args(const GMat &W, const float *x, const float *gains, float eps, const float *bias, float *y,
                   const GCursor *cur, int m = 1, int xs = 0) {
  GemvArgs a{};
  a.m = m;
  a.xs = xs;
  a.W = W;
  a.x = x;
  a.gains = gains;
  a.eps = eps;
  a.bias = bias;
  a.y = y;
  a.cur = cur;
  return a;
}

}  // namespace

bool g_kind_supported(int kind, int group) {
  switch (kind) {
  case MLLM_F32:
  case MLLM_F16:
  case MLLM_BF16:
  case MLLM_Q8: return true;
  case MLLM_Q8G32: return group == 32;
  case MLLM_Q4: return group >= 8 && group % 8 == 0;
  default: return false;
  }
}

int g_gemv(const GMat &W, const float *x, float *y, hipStream_t s) {
  MLLM_CHECK(g_kind_supported(W.kind, W.group) && W.cols % 8 == 0 && (W.kind != MLLM_Q4 || W.cols % W.group == 0),
             "matrix storage %d (group %d, %d columns) unsupported", W.kind, W.group, W.cols);
  MLLM_CHECK(W.cols <= 16000, "%d columns exceed 16000", W.cols);
  launch_gemv<G_STORE, GN_NONE>(gemv_args(W, x, nullptr, 0.f, nullptr, y, nullptr), s);
  MLLM_HIP(hipGetLastError());
  return 0;
}

int g_head(const GArgs &A, const float *x, int m, hipStream_t s) {
  GemvArgs f = gemv_args(A.lm, x, A.norm_f, A.eps, nullptr, A.logits, A.cur, m, A.D);
  f.lm = 1;
  if (A.arch == 1)
    launch_gemv<G_STORE, GN_LN>(f, s);
  else
    launch_gemv<G_STORE, GN_RMS>(f, s);
  hipLaunchKernelGGL(k_g_argmax, dim3(m), dim3(GAT), sizeof(int) * (34 + (size_t)A.max_seq), s, A);
  MLLM_HIP(hipGetLastError());
  return 0;
}

int g_step(const GArgs &A, bool lm, int m, hipStream_t s) {
  const bool gpt2 = A.arch == 1;
  const GCursor *cur = A.cur;
  hipLaunchKernelGGL(k_g_embed, dim3(m), dim3(GT), 0, s, A);
  const int nsplit = (A.max_seq + GSPLIT - 1) / GSPLIT;
  for (int li = 0; li < A.L; ++li) {
    const GLayer &w = A.layers[li];
    if (!(w.dbg & 1)) {
      GemvArgs q = gemv_args(w.qkv, A.x, w.n1, A.eps, w.qkv_b, A.qkv, cur, m, A.D);
      if (gpt2)
        launch_gemv<G_STORE, GN_LN>(q, s);
      else
        launch_gemv<G_STORE, GN_RMS>(q, s);
      if (m > 1) hipLaunchKernelGGL(A.kv_fp16 ? k_g_kv<true> : k_g_kv<false>, dim3(A.NKV, m), dim3(GHD), 0, s, A, li);
      hipLaunchKernelGGL(A.kv_fp16 ? k_g_attn<true> : k_g_attn<false>, dim3(A.NH, nsplit, m), dim3(GAW * 64), 0, s, A, li);
      GemvArgs o = gemv_args(w.proj, A.attp, nullptr, 0.f, w.proj_b, A.x, cur, m, A.NH * nsplit * GAPS);
      o.nsplit_max = nsplit;
      launch_gemv<G_RESID, GN_SPLITS>(o, s);
    }
    if (!(w.dbg & 2)) {
      if (gpt2) {
        launch_gemv<G_GELU, GN_LN>(gemv_args(w.w1, A.x, w.n2, A.eps, w.fc_b, A.h, cur, m, A.D), s);
      } else {
        GemvArgs u = gemv_args(w.w1, A.x, w.n2, A.eps, nullptr, A.h, cur, m, A.D);
        u.W3 = w.w3;
        launch_gemv<G_SWIGLU, GN_RMS>(u, s);
      }
      launch_gemv<G_RESID, GN_NONE>(gemv_args(w.w2, A.h, nullptr, 0.f, w.mproj_b, A.x, cur, m, A.FF), s);
    }
  }
  if (lm) return g_head(A, A.x, m, s);
  MLLM_HIP(hipGetLastError());
  return 0;
}

}  // namespace mllm
