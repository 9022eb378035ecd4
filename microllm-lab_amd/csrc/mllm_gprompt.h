// mllm_gprompt.h -- batched prompts (infer.js:553-577 forwardPrompt) of the
// models that run the kind-generic decode step: matrices in any storage, a
// chunk of prompt tokens through each layer as a few kernels on the bf16
// matrix cores, K and V written to the cache.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mllm_generic.h"

namespace mllm {

// The tiled copy of a matrix that the prompt GEMMs read: np bf16 planes of
// its values (per-row Q8: of its integers, rs the rows' scales), see gp_tile.
struct GpMat {
  const uint8_t *t;
  const float *rs;
  int rows, cols, np;
};

struct GpLayer {
  GpMat qkv, proj, w1, w3, w2;                   // gpt2: w1 = mlp.fc, w2 = mlp.proj, no w3
  const float *n1, *n2;                          // RMS gains; gpt2: LayerNorm gamma || beta
  const float *qkv_b, *proj_b, *fc_b, *mproj_b;  // gpt2 biases (proj_b / mproj_b may be null)
};

struct GpArgs {
  int arch, L, D, NH, NKV, FF, max_seq, kv_fp16, rope_dim;
  float eps, attn_scale;
  const GpLayer *layers;  // host array of L layers
  GMat emb;               // tied lm_head: the embedding rows
  const float *wpe, *sf, *rope_cos, *rope_sin;
  void *kv;  // [L][2][NKV][max_seq][64], f32 or f16
  // work buffers for up to tc tokens
  int tc;
  int32_t *ids;  // [tc]
  float *x;      // [tc][D] residual stream
  float *q;      // [tc][D] roped queries
  float *ss;     // [tc][D / 64] sums of squares of the residual's 64-column blocks
  uint8_t *pxa;  // planes (mllm_planes.h) of a GEMM's normalised input [tc][D]
  uint8_t *pxo;  // of the attention output [tc][D]
  uint8_t *pxh;  // of the MLP activation [tc][FF]
};

// Planes that hold a storage kind's values: bf16 and per-row Q8 integers 1,
// f16 2 (both exact); f32 3 (exact); Q8 group-32 and Q4 3 (the de-quantised
// float32 value).
int gp_planes(int kind);

// Tiled copy: for row tile rt (32 rows) and group g of 32 columns, plane p and
// half m: 64 lanes of 16 bytes, lane 32 hh + j holding columns 16m + 8hh .. +7
// of row 32 rt + j (the tokens' own order).  rows and cols multiples of 32.
size_t gp_tiled_bytes(int rows, int cols, int np);
int gp_tile(const GMat &W, int np, void *dst, GpMat *out, hipStream_t s);

// Shapes the kernels take: at most 4 query heads per KV head, d_ff a multiple
// of 64.
bool gp_supported(const GpArgs &A);

// Bytes of work buffers for tc tokens (one allocation, carved by gp_carve).
size_t gp_buffer_bytes(const GpArgs &A, int tc);
void gp_carve(GpArgs &A, void *base, int tc);

// Once per device before the first gp_layers: the kernels' LDS limits.
int gp_init();

// Tokens ids[0 .. n) at positions pos0 .. through every layer (n <= tc).
// With `last` the last token's residual row leaves every layer and *row is
// where it lies; otherwise the last layer stops after its K and V.
int gp_layers(const GpArgs &A, const int32_t *ids, int n, int pos0, bool last, const float **row, hipStream_t s);

}  // namespace mllm
