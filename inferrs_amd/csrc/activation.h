// The activations of a feed-forward without a gate, of values that are stored: 1 SiLU, 2 GELU in its tanh form, 3 the exact GELU.
#pragma once

#include "common.h"

// The exact GELU of a value that is stored in 16 bits: max(z, 0) - |z| / 2 erfc(|z| / sqrt 2), erfc(|z| / sqrt 2) = exp(-z^2 / 2) t P(t),
// t = 1 / (1 + 0.26 |z|), P a polynomial fitted to exp(z^2 / 2) erfc(|z| / sqrt 2) / t in 64 bits up to |z| = 14 (least squares, reweighted
// towards the smallest largest relative error: 2.5e-8).  z^2 is exact, no branch, and nothing cancels: of all bfloat16 values those above -4 give
// the bits of the formula with erff, those below are right where 1 + erff had lost them (a third of the value off between -6 and
// -4 in the mean).  erff's two branches, which a wave takes both, were what bounded the pass.  An infinity gives what the formula gives.
__device__ __forceinline__ float gelu_for_bf16(float z) {
    const float a = fminf(fabsf(z), 64.0f);                  // (beyond: erfc is 0; a product of infinity and 0 would be no number)
    const float t = __builtin_amdgcn_rcpf(fmaf(0.26f, a, 1.0f));
    float p = 0.06100985f;
    p = fmaf(p, t, -0.30565804f);
    p = fmaf(p, t, 0.50298333f);
    p = fmaf(p, t, -0.30189878f);
    p = fmaf(p, t, 0.32189628f);
    p = fmaf(p, t, 0.10205514f);
    p = fmaf(p, t, 0.20606056f);
    p = fmaf(p, t, 0.2060335f);
    p = fmaf(p, t, 0.20751812f);
    return fmaf(0.5f, z, 0.5f * fabsf(z)) - 0.5f * a * t * p * __builtin_amdgcn_exp2f(a * a * -0.72134752f);
}
template <typename T>
__device__ __forceinline__ float act_stored(float z, int act) {
    if (act != 3) return gate_act(z, act);
    if constexpr (sizeof(T) == 2) return gelu_for_bf16(z);
    else return 0.5f * z * (1.0f + erff(z * 0.7071067811865476f));
}
