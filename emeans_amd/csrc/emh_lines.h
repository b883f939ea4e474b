// The one-pass screens' operands (k_screen5): rows or centroids rounded once
// to fp16, in lines, shared by the kernels that write them (k_lines).
//
// A matrix is scaled by one power of two s (scale[0]; scale[1] = 1 / s) that
// brings its largest sampled element to 2^7 .. 2^8, and cut into slabs of 32
// dimensions (dimensions past d are zero), each a 64-byte line of fp16
// values h(s x), rounded to nearest even, in order. Lines are stored
// slab-major: slab j of row g of an n-row matrix at (j n + g) 64 bytes.
//
// The centroids' side (kNN: the data's) is rounded as its difference from one
// vector m, the mean of sampled rows where those have one that matters, else
// zero (k_scales). x.c = x.(c - m) + x.m, and x.m is the same for every
// centroid of a row, so the screen's keys are the row's keys less a constant
// and order its centroids alike, while the error falls from |x||c| to
// |x||c - m|: rows that share most of their length (unit rows with a mean
// cosine of 0.92: |c - m| = 0.29 |c|) would otherwise have more near-ties than
// their lists hold.
//
// A row's rounding residual r = |s x - h(s x)| is kept beside |x|^2: the
// screen's error bound follows from Cauchy-Schwarz on the residuals that the
// rounding really left (about 0.4 of the worst case of 2^-11 |x| on ordinary
// values), and values below fp16's normal range, or above 65504 (h infinite,
// r infinite, the row or every row goes to the exact scan) need no rule of
// their own. Where nothing is far out of range the scale is exact, so it
// changes no bound.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace emh {

constexpr int LINE_BYTES = 64;  // one row's 32 dimensions (half a cache line)
constexpr int LINE_DIMS = 32;
// Bytes of n rows' lines, with room for a tile's rows past the last (which the
// screen reads, and never uses).
inline size_t lines_bytes(size_t n, size_t d) {
  return (n * ((d + LINE_DIMS - 1) / LINE_DIMS) + 256) * LINE_BYTES;
}

typedef _Float16 v4h_l __attribute__((ext_vector_type(4)));

// A mean's floats: zeros past d, so that whole lines can read it, then whether
// it is one (1) or all zeros (0).
__host__ __device__ inline size_t mean_flag(size_t d) {
  return (d + LINE_DIMS - 1) / LINE_DIMS * LINE_DIMS;
}
inline size_t mean_floats(size_t d) { return mean_flag(d) + 4; }

// Four scaled values rounded to fp16 (8 bytes of a line); res += the squares
// of what the rounding left (exact differences: v and h are multiples of one
// another's ulp).
__device__ __forceinline__ uint2 line_quad(float4 v, float s, float& res) {
  const float e[4] = {v.x * s, v.y * s, v.z * s, v.w * s};
  v4h_l h4;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const _Float16 h = (_Float16)e[t];
    h4[t] = h;
    const float r = e[t] - (float)h;
    res = fmaf(r, r, res);
  }
  return __builtin_bit_cast(uint2, h4);
}

// The one-pass screens' bound E on |screen key - (exact key + const)| for one
// row, the constant x.m (L2: 2 x.m) the same for all its centroids (see
// screen_bound in emh_select.h for the terms that both share). xn = |x|^2 and
// xr = |s x - h(s x)|^2 of the row, cmax2, vmax2, rmax2 and cnmax the
// centroids' largest |c|^2, |v|^2 (v = c - m), residual and given norm (f32
// sums in any order, relative error <= gamma_d), isx and isc the inverse
// scales. With rx, rc the residuals in x's and c's units,
//   |x.v - xh.vh| <= |x - xh||v| + |xh||v - vh| <= rx |v| + (|x| + rx) rc;
//   c - m rounded to f32: u |x||v|;
//   the check's fma chain: gamma_d |x||c|;
//   the MFMA chain of M = 2 ceil(d / 32) MFMAs, each within 16 u of its
//   terms' magnitudes (products of two fp16 values are exact in f32):
//   gamma(16 M) |xh||vh|;
//   underflow: (3 d + M) 2^-124.
// The keys carry a 7-bit column tag in their low mantissa bits: at most 127
// ulp < 2^-16 |key|, |key| <= |c|^2 + 2 |xh||vh| (L2), |xh||vh| (IP), a few
// roundings apart, plus 127
// subnormal ulps.
// A sum of squares that underflows loses at most d 2^-149 (uf). Not finite
// (an element beyond fp16's range, NaN, a key that may overflow f32): NaN, which
// settles nothing.
// edot_out: the dot term alone.
__device__ __forceinline__ float screen_bound_lines(float xn, float xr, float cmax2, float vmax2,
                                                    float rmax2, float cnmax, float isx, float isc,
                                                    int d, bool l2, float* edot_out) {
  const float u = 5.9604645e-08f;  // 2^-24
  const float du = (float)d * u;
  const float g = du / (1.0f - du);
  const float uf = (float)d * 1.4012985e-45f;  // d 2^-149
  const float xa = sqrtf(xn + uf) * (1.0f + g), ca = sqrtf(cmax2 + uf) * (1.0f + g);
  const float va = sqrtf(vmax2 + uf) * (1.0f + g);
  const float rx = sqrtf(xr + uf) * (1.0f + g) * isx, rc = sqrtf(rmax2 + uf) * (1.0f + g) * isc;
  const float m = (float)(2 * ((d + LINE_DIMS - 1) / LINE_DIMS));
  const float mu = 16.0f * m * u;
  const float gm = mu / (1.0f - mu);
  const float S = xa * ca;
  const float H = (xa + rx) * (va + rc);
  float edot = g * S + (rx + u * xa) * va + (xa + rx) * rc + gm * H +
               (float)(3 * d + (int)m) * 4.7019774e-38f;
  // Few dimensions come close to the Cauchy-Schwarz terms (0.62 of them over
  // 24,616 listed pairs at d = 36, 0.2 at 768): half as much again below 64
  // keeps the bound at twice what is seen, at any width.
  if (d < 64) edot = 1.5f * edot;
  if (!(edot < INFINITY)) edot = __builtin_nanf("");
  *edot_out = edot;
  float e = l2 ? 2.0f * edot + 2.0f * u * (cnmax + 2.0f * fmaxf(S, H)) : edot;
  e += 1.5268e-5f * (l2 ? cnmax + 2.0f * H : H) + 1.8e-43f;
  e *= 1.015625f;  // the rounding of these few operations
  return e < INFINITY ? e : __builtin_nanf("");
}

}  // namespace emh
