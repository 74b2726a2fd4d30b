// Kernel value of one pair from its scaled squared distance (kernel_scale()),
// shared by the per-pair kernels of matvec.hip and direct.hip.
#pragma once

#include "matvec.h"

namespace mgp {

constexpr float kM52A = 0.69314718055994530942f;                     // ln 2
constexpr float kM52B = 0.69314718055994530942f * 0.69314718055994530942f / 3.0f;

// Kernel value from the scaled squared distance s (see kernel_scale()).
// clampv = the exponent limit exp2_limit(kind, ard) (kExp2Clamp, from
// clamp_reg() in hot loops, for the Matern-3/2 and 5/2 kernels; the point
// set's exp2_limit for Matern-1/2; RBF has none).
template <int KIND>
__device__ __forceinline__ float kval(float s, float clampv = kExp2Clamp) {
  if constexpr (KIND == KIND_RBF) {
    // os * exp(-0.5 r^2) = os * 2^-max(s, 0) (the max only absorbs Gram-form
    // rounding below zero; the reference does not clamp the RBF exponent)
    return __builtin_amdgcn_exp2f(-fmaxf(s, 0.0f));
  } else if constexpr (KIND == KIND_MATERN12) {
    // os * exp(-r) (isotropic) or os * exp(max(-r, -20)) (ARD),  u = r log2 e
    const float u = __builtin_amdgcn_sqrtf(fabsf(s));
    return __builtin_amdgcn_exp2f(-fminf(u, clampv));
  } else if constexpr (KIND == KIND_MATERN32) {
    // os * (1 + sqrt3 r) * exp(max(-sqrt3 r, -20)),  u = sqrt3 r log2 e
    const float u = __builtin_amdgcn_sqrtf(fabsf(s));
    return fmaf(u, kLn2, 1.0f) * __builtin_amdgcn_exp2f(-fminf(u, clampv));
  } else {
    // os * (1 + sqrt5 r + 5/3 r^2) * exp(max(-sqrt5 r, -20)),  u = sqrt5 r log2 e
    // sqrt(|s|): s < 0 only from Gram-form rounding of a near-zero distance,
    // where |s| and max(s, 0) agree to the rounding error (dk/du = 0 at u = 0);
    // the abs is a free source modifier of v_sqrt_f32.
    const float u = __builtin_amdgcn_sqrtf(fabsf(s));
    // min(u, C) kept opaque so that the negation is not rewritten into
    // max(-u, -C) + v_xor but lands on v_exp_f32 as a source modifier.
    float m = fminf(u, clampv);
    asm("" : "+v"(m));
    const float e = __builtin_amdgcn_exp2f(-m);
    const float p = fmaf(u, fmaf(u, kM52B, kM52A), 1.0f);
    return p * e;
  }
}

}  // namespace mgp
