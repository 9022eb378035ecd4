// mllm_planes.h -- float32 rows as three bf16 planes for the matrix cores.
//
// A value x is split by rounding to nearest: p0 = bf16(x), p1 = bf16(x - p0),
// p2 = bf16(x - p0 - p1).  Each plane takes 8 significant bits and both
// differences are exact in float32, so p0 + p1 + p2 is x itself (24 bits)
// except below 2^-110 or so, where the last plane leaves the exponent range.
// bf16 has float32's exponents: no row scale is needed, so a kernel that has
// only some of a row's columns can write their planes.
//
// Tokens are stored in the operand order of v_mfma_f32_32x32x16_bf16, tile by
// tile: for 32 tokens and a group of 32 columns, plane p, half m (columns
// 16m .. 16m+15 of the group) are 64 lanes of 16 bytes, lane 32 hh + j holding
// columns 16m + 8hh .. +7 of token j.  So a wave reads one operand as 1 KiB of
// consecutive bytes, and eight columns of a token are one 16-byte store.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace mllm {

constexpr int BPX = 6 * 1024;  // bytes per (32-token tile, group of 32 columns): 3 planes x 2 halves x 64 lanes x 16

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2fl __attribute__((ext_vector_type(2)));

// The planes of two values, packed (the first in the low half).  The first
// plane of a finite value is taken from the value cut to bf16's largest, so that
// one past it keeps finite planes.  An infinity or NaN is itself in the first
// plane and NaN in the others: a sum of first-plane products that is not finite
// is the result, without the other planes' products.
__device__ __forceinline__ float bf16_cut(float v) {
  constexpr float M = 3.3895313892515355e38f;
  return fabsf(v) < INFINITY ? __builtin_amdgcn_fmed3f(v, -M, M) : v;
}
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2fl){a, b}, v2bf));  // nearest even
}
__device__ __forceinline__ void bf16_split2(float a, float b, uint32_t (&p)[3]) {
  p[0] = bf16_pair(bf16_cut(a), bf16_cut(b));
  a -= __uint_as_float(p[0] << 16);
  b -= __uint_as_float(p[0] & 0xffff0000u);
  p[1] = bf16_pair(a, b);
  a -= __uint_as_float(p[1] << 16);
  b -= __uint_as_float(p[1] & 0xffff0000u);
  p[2] = bf16_pair(a, b);
}

// Columns 4c .. 4c+3 (v) of token j of a tile (its group 0 at `tile`).
__device__ __forceinline__ void planes_store4(uint8_t *tile, int j, int c, const float (&v)[4]) {
  uint32_t a[3], b[3];
  bf16_split2(v[0], v[1], a);
  bf16_split2(v[2], v[3], b);
  uint8_t *o = tile + (size_t)(c >> 3) * BPX + ((c >> 1) & 3) * 512 + j * 16 + (c & 1) * 8;
#pragma unroll
  for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2 *>(o + 2048 * p) = make_uint2(a[p], b[p]);
}

}  // namespace mllm
