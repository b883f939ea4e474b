// The split-operand layout of rows for the fp16 two-pass screen (k_screen4),
// shared by the kernels that write it (k_halves, and k_ema, k_split_fused and
// the small-batch update for the centroids they move).
//
// A row is cut into slabs of 32 dimensions (dimensions past d are zero), each
// 128 bytes, one cache line, stored slab-major: slab j of row g of an n-row
// matrix at (j n + g) 128 bytes. A slab row holds eight 16-byte chunks: for
// MFMA step kk = 0, 1 (dimensions 16 kk .. 16 kk + 15), chunks 4 kk and
// 4 kk + 1 are the hi halves of its two 8-dimension groups and chunks
// 4 kk + 2 and 4 kk + 3 their lo halves, rounded to nearest even (x - hi is
// exact in f32): hi = fp16(x), lo = fp16(x - hi): |x - hi| <= 2^-11 |x| +
// 2^-25 and |x - hi - lo| <= 2^-22 |x| + 2^-25 (1 + 2^-11) for |x| < 65520
// (rows hi + lo, centroids hi).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "emh_internal.h"
#include "emh_lines.h"

namespace emh {

constexpr int SLAB_BYTES = 128;  // one row's 32 dimensions (one cache line)

typedef _Float16 v4h_h __attribute__((ext_vector_type(4)));

// Byte offset, within a slab row, of the hi quad of dimensions 4 c4 .. 4 c4 + 3
// of the slab (c4 = 0 .. 7); the lo quad sits 32 bytes later.
__device__ __forceinline__ int quad_hi_offset(int c4) {
  const int c8 = c4 >> 1;  // the 8-dimension group
  return 16 * (4 * (c8 >> 1) + (c8 & 1)) + 8 * (c4 & 1);
}

// The hi and lo halves of four values, as two 8-byte quads.
__device__ __forceinline__ void split_quad(float4 v, uint2& hi, uint2& lo) {
  const float e[4] = {v.x, v.y, v.z, v.w};
  v4h_h h4, l4;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const _Float16 h = (_Float16)e[t];
    h4[t] = h;
    l4[t] = (_Float16)(e[t] - (float)h);
  }
  hi = __builtin_bit_cast(uint2, h4);
  lo = __builtin_bit_cast(uint2, l4);
}

// Dimensions col .. col + 3 (col % 4 == 0, those past d zero) of row j of k
// rows. Lines: (the squares of the quad's difference from the mean, the
// residual its rounding left).
__device__ __forceinline__ float2 put_quad(const CentsOut& o, size_t k, size_t j, size_t col,
                                           float4 v) {
  if (o.scale) {
    const float4 m = *reinterpret_cast<const float4*>(o.scale + MEAN_AT + col);  // (zeros past d)
    v = make_float4(v.x - m.x, v.y - m.y, v.z - m.z, v.w - m.w);
    float res = 0.f;
    const uint2 q = line_quad(v, o.scale[0], res);
    *reinterpret_cast<uint2*>(o.cs + ((col / LINE_DIMS) * k + j) * LINE_BYTES +
                              2 * (col % LINE_DIMS)) = q;
    return make_float2(fmaf(v.w, v.w, fmaf(v.z, v.z, fmaf(v.y, v.y, v.x * v.x))), res);
  }
  uint2 hi, lo;
  split_quad(v, hi, lo);
  char* p = o.cs + ((col >> 5) * k + j) * SLAB_BYTES + quad_hi_offset((int)(col & 31) >> 2);
  *reinterpret_cast<uint2*>(p) = hi;
  *reinterpret_cast<uint2*>(p + 32) = lo;
  return make_float2(0.f, 0.f);
}

// The figures of a row's quads into its two sums in LDS: eight lanes, which
// hold quads of one row, first add theirs up.
__device__ __forceinline__ void add_quad(float2 r, float* dif, float* res) {
#pragma unroll
  for (int m = 1; m < 8; m <<= 1) {
    r.x += __shfl_xor(r.x, m, 64);
    r.y += __shfl_xor(r.y, m, 64);
  }
  if ((threadIdx.x & 7) == 0) {
    atomicAdd(dif, r.x);
    atomicAdd(res, r.y);
  }
}

}  // namespace emh
