// mllm_kinds.h -- reading a matrix in any storage the models carry (f32,
// f16, bf16, per-row Q8, Q8 group-32, Q4 of any group that is a multiple of
// 8), eight columns at a time: shared by the kind-generic decode step and the
// batched prompts of the same models.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mllm.h"
#include "mllm_generic.h"

namespace mllm {

__device__ __forceinline__ float f16_bits(uint32_t h) { return __half2float(__ushort_as_half((unsigned short)h)); }
__device__ __forceinline__ float bf16_bits(uint32_t h) { return __uint_as_float(h << 16); }

// Columns 8c .. 8c+7 of row r as floats (w) and the chunk's scale (Q8
// group-32 and Q4: the group's; 1 otherwise -- per-row Q8 scales the row's sum).
__device__ __forceinline__ float load8(const GMat &W, int r, int c, float (&w)[8]) {
  const size_t e0 = (size_t)r * W.cols + 8 * (size_t)c;
  switch (W.kind) {
  case MLLM_F32: {
    const float4 *p = reinterpret_cast<const float4 *>(static_cast<const float *>(W.w) + e0);
    const float4 a = p[0], b = p[1];
    w[0] = a.x, w[1] = a.y, w[2] = a.z, w[3] = a.w, w[4] = b.x, w[5] = b.y, w[6] = b.z, w[7] = b.w;
    return 1.f;
  }
  case MLLM_F16:
  case MLLM_BF16: {
    const uint4 u = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(W.w) + e0);
    const uint32_t p[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w[2 * k] = W.kind == MLLM_F16 ? f16_bits(p[k] & 0xffffu) : bf16_bits(p[k] & 0xffffu);
      w[2 * k + 1] = W.kind == MLLM_F16 ? f16_bits(p[k] >> 16) : bf16_bits(p[k] >> 16);
    }
    return 1.f;
  }
  case MLLM_Q8:
  case MLLM_Q8G32: {
    const uint2 u = *reinterpret_cast<const uint2 *>(static_cast<const int8_t *>(W.w) + e0);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w[k] = (float)(int8_t)(u.x >> (8 * k));
      w[4 + k] = (float)(int8_t)(u.y >> (8 * k));
    }
    return W.kind == MLLM_Q8G32 ? W.s[(size_t)r * (W.cols >> 5) + (c >> 2)] : 1.f;
  }
  default: {  // MLLM_Q4: byte k holds element 2k (low nibble) and 2k + 1, stored as q + 8
    const uint32_t u = *reinterpret_cast<const uint32_t *>(static_cast<const uint8_t *>(W.w) + e0 / 2);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w[2 * k] = (float)((int)((u >> (8 * k)) & 15u) - 8);
      w[2 * k + 1] = (float)((int)((u >> (8 * k + 4)) & 15u) - 8);
    }
    return W.s[(size_t)r * (W.cols / W.group) + (8 * c) / W.group];
  }
  }
}

}  // namespace mllm
