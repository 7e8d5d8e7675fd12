// f32 products on the f16 matrix cores: each operand goes in as two f16 parts,
// x * 2^s = hi + lo, and a dot product is hi*hi + hi*lo + lo*hi summed in f32
// (v_mfma_f32_32x32x16_f16). Shared by the flat search's and k-means'
// approximate distances, whose results are certified and recomputed exactly.
//
// Why: an f32 MFMA multiplies at 157 TFLOP/s, an f16 one at 16 times that, so
// three f16 products cost 3/16 of the f32 pass. Nothing is lost against it:
//   - hi + lo holds x * 2^s to one unit of f32's last place (24 significant
//     bits, of which the two 11-bit parts and lo's sign miss at most the last
//     one), and the products themselves are exact in f32;
//   - the missing lo*lo term is below 2^-22 of |x_i q_i|;
//   - the accumulator is rounded twice per 16 dimensions and product instead
//     of once per dimension.
// Measured against 64-bit dot products (rms error over |q||x|, in units of
// 2^-24; f32 MFMA -> this): d = 64: 1.94 -> 1.14 and 0.30 -> 0.24, d = 128:
// 2.67 -> 1.58 and 0.30 -> 0.21, d = 768: 6.81 -> 4.15 and 0.30 -> 0.19
// (clustered and independent rows). Below 64 dimensions the split's own
// rounding is no longer hidden by the sum's, so those keep the f32 pass.
//
// Error of one dot product of d terms, any order, against |q||x| in units of
// 2^-24: an MFMA adds the products in two groups of eight onto the
// accumulator, nine terms aligned to the largest and cut at most 2^-24 of it
// below, then one rounding, so 10 per group and 20 per MFMA: 3.75 D for the
// 3 D / 16 of them, D being d rounded up to a multiple of 16 (those past it
// add zeros to the accumulator, which is exact). (Measured over 10^8 MFMAs
// with operands of up to 28 binades' spread, single ones are within 8.5.) The
// parts miss at most 2^-23 of each operand, 2 units each, and the missing
// lo*lo is below 4: 8 in all.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace pxg {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));

// Dimensions from which the split product is at least as accurate as the f32
// MFMA's.
constexpr uint32_t SPLIT_MIN_DIM = 64;

// The power of two that takes a norm to [2^14, 2^15), so that every part is
// inside f16's range (what rounds to a subnormal part is below 2^-38 of the
// norm); 1 for zero.
__host__ __device__ inline float split_scale(float norm) {
  if (norm == 0.0f) return 1.0f;
  int ex;
  (void)frexpf(norm, &ex);
  return ldexpf(1.0f, 15 - ex);
}
// Norms whose scales stay normal floats. Two such scales can multiply past f32
// (2^75 each), so they are divided by one after the other, never multiplied.
__host__ __device__ inline bool split_norm_ok(float norm) { return norm >= 0x1p-60f && norm <= 0x1p+60f; }

// One x * s as its two f16 parts (the fma forms are exact: s is a power of
// two, and x * s - hi has at most 13 bits).
__device__ __forceinline__ void split_f16(float x, float s, _Float16& hi, _Float16& lo) {
  hi = (_Float16)__builtin_fmaf(x, s, 0.0f);
  lo = (_Float16)__builtin_fmaf(x, s, -(float)hi);
}

}  // namespace pxg
