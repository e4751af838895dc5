// The gated units at the end of the fused gate/up products.
#pragma once
#include "common.h"

// silu for the epilogues whose result is rounded to bfloat16 at once: the hardware's exp2 and reciprocal (about an
// ulp of float each) instead of the library's exp and an exact division, a fifth of the instructions; the ends of
// the range come out right (exp2 = inf gives -0, exp2 = 0 gives g). Of all 65,280 finite bfloat16 gates one comes out a bfloat16
// step from the rounded 64-bit result, and results below 1e-36 come out as 0 (from -87.5 down; by exact division from -89).
__device__ __forceinline__ float silu_for_bf16(float g) {
  return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f));
}

// Of one output's gate and up, float: T(T(silu(T(gate))) * T(up)). With `limit` > 0 the unit is the clamped one instead:
// g = min(gate, limit), u = clamp(up, -limit, limit), T(g * sigmoid(alpha g) * (u + 1)), rounded once. With `relu` it is
// T(max(gate, 0) * up), also rounded once.
struct GateAct {
  float limit = 0.f, alpha = 0.f;
  int relu = 0;
};
__device__ __forceinline__ float clamped_unit(float gate, float up, const GateAct& act) {
  const float gc = fminf(gate, act.limit), uc = fminf(fmaxf(up, -act.limit), act.limit);
  return gc * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(gc * act.alpha * -1.4426950408889634f)) * (uc + 1.f);
}
__device__ __forceinline__ bf16_t gate_unit(float gate, float up, const GateAct& act) {
  return act.relu            ? float_to_bf16(fmaxf(gate, 0.f) * up)
         : act.limit > 0.f ? float_to_bf16(clamped_unit(gate, up, act))
                           : float_to_bf16(rounded_as<bf16_t>(silu_for_bf16(rounded_as<bf16_t>(gate))) * rounded_as<bf16_t>(up));
}
