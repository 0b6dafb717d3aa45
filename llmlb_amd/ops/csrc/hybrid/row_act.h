// What becomes of a product's sums before they are stored: a launch less
// than a kernel of its own, and a pass over memory less.  The sum is rounded
// to bf16 first, as where it is stored for that kernel.  With two matrices,
// gate and up, the rows of up begin at row ``up`` of the weight.
#pragma once
#include "mfma.h"

enum RowKind { PLAIN, RELU2, GELU, SWIGLU, CLAMPED, CAPPED };
struct RowAct {
  int kind;
  int up;      // SWIGLU, CLAMPED: the first row of up
  float a, b;  // CLAMPED: limit, sharpness; CAPPED: cap (0: none)
};
// n / (1 + e), e not below 0.  What the reciprocal's quotient leaves over is
// divided once more (Markstein), in half the instructions of a division, which
// nothing in an epilogue hides: 16384 rows, gate and up of 28672 x 4096 2594 us
// with divisions, 2550 this way, 2530 by the reciprocal alone, which is 1.5
// units in the last place off; of 5632 x 1024 167, 160, 154.  Of 65280 gates
// beside 130 numbers each no result differs from the division's.  Both sides
// are a fourth: the hardware's reciprocal of numbers above 2^126 is zero.
__device__ __forceinline__ float row_ratio(float n, float e) {
  const float d = fmaf(0.25f, e, 0.25f), m = 0.25f * n;
  const float r = __builtin_amdgcn_rcpf(d), q = m * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, m), r, q), d, m);
}
// gelu, its tanh form: z / (1 + exp(-2 k (z + c z^3))), k = sqrt(2 / pi).  z is a
// bf16 number, and so is what becomes of the result: of all of them none
// differs from gelu_tanh_fast's.
__device__ __forceinline__ float row_gelu(float z) {
  constexpr float k = -2.f * 0.7978845608028654f * LOG2E;
  const float t = z * (k + k * 0.044715f * (z * z));
  return z * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(t));
}
__device__ __forceinline__ float row_act(const RowAct& act, float z) {
  if (act.kind == RELU2) {
    z = fmaxf(z, 0.f);
    return z * z;
  }
  if (act.kind == GELU) return row_gelu(z);
  if (act.kind == CAPPED && act.a > 0.f) return act.a * tanhf(z / act.a);
  return z;
}
__device__ __forceinline__ float row_gate(const RowAct& act, float g,
                                          float u) {
  if (act.kind == SWIGLU) return row_ratio(g, __expf(-g)) * u;
  g = fminf(g, act.a);
  u = fminf(fmaxf(u, -act.a), act.a);
  return row_ratio(g, __expf(-act.b * g)) * (u + 1.f);
}
