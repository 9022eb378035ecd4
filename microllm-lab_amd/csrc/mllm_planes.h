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
#include <stdint.h>

namespace mllm {

constexpr int BPX = 6 * 1024;  // bytes per (32-token tile, group of 32 columns): 3 planes x 2 halves x 64 lanes x 16

// Bits of the nearest bf16 (ties to even); a finite value past bf16's largest
// is cut instead, so that the planes of a finite value stay finite.
__device__ __forceinline__ uint32_t bf16_rne(float x) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t r = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
  return (r & 0x7f80u) == 0x7f80u ? u >> 16 : r;
}
__device__ __forceinline__ void bf16_split3(float x, uint32_t &p0, uint32_t &p1, uint32_t &p2) {
  p0 = bf16_rne(x);
  // an infinity or NaN is all in the first plane
  const float r1 = (p0 & 0x7f80u) == 0x7f80u ? 0.f : x - __uint_as_float(p0 << 16);
  p1 = bf16_rne(r1);
  p2 = bf16_rne(r1 - __uint_as_float(p1 << 16));
}

// Columns 8c .. 8c+7 (v) of token j of tile base `tile` (its group 0).
__device__ __forceinline__ void planes_store8(uint8_t *tile, int j, int c, const float (&v)[8]) {
  uint32_t p0[8], p1[8], p2[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) bf16_split3(v[e], p0[e], p1[e], p2[e]);
  uint8_t *o = tile + (size_t)(c >> 2) * BPX + ((c >> 1) & 1) * 1024 + (c & 1) * 512 + j * 16;
  *reinterpret_cast<uint4 *>(o) =
      make_uint4(p0[0] | p0[1] << 16, p0[2] | p0[3] << 16, p0[4] | p0[5] << 16, p0[6] | p0[7] << 16);
  *reinterpret_cast<uint4 *>(o + 2048) =
      make_uint4(p1[0] | p1[1] << 16, p1[2] | p1[3] << 16, p1[4] | p1[5] << 16, p1[6] | p1[7] << 16);
  *reinterpret_cast<uint4 *>(o + 4096) =
      make_uint4(p2[0] | p2[1] << 16, p2[2] | p2[3] << 16, p2[4] | p2[5] << 16, p2[6] | p2[7] << 16);
}

}  // namespace mllm
