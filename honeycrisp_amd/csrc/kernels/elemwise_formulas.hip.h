// Pieces of the element-wise formulas that more than one code object needs: kernels that take over
// the work of an element-wise kernel when a recording merges it into its producer (GELU in a GEMM
// epilogue, exp after a log-softmax) must produce the bits of the separate kernel. Every file
// that includes this is built with -ffp-contract=off (the reference never fuses a * b + c).
#pragma once

// Formulas of ElemwiseOp.apply (Elemwise.swift:44-183), same expression trees.
__device__ __forceinline__ float safe_sigmoid(float x) {
  if (x < -20.0f) return 0.0f;
  if (x > 20.0f) return 1.0f;
  return 1.0f / (1.0f + expf(-x));
}
__device__ __forceinline__ float safe_tanh(float x) { return 2.0f * safe_sigmoid(2.0f * x) - 1.0f; }

// The same for results that are rounded to fp16 (11 significant bits): the hardware's exp2 and
// reciprocal (about 1 ulp of fp32 each) instead of the library's expf and an IEEE division.
// With the library routines an fp16 GELU is bound by the vector ALU (8 elements per 16-byte
// load), not by memory.
__device__ __forceinline__ float exp_hw(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }
__device__ __forceinline__ float sigmoid_hw(float x) {
  // (computed first, then selected: no branch per element, so the elements of a vector overlap)
  const float inside = __builtin_amdgcn_rcpf(1.0f + exp_hw(-x));
  return x < -20.0f ? 0.0f : (x > 20.0f ? 1.0f : inside);
}
// GELU for results that are rounded to fp16: (1 + tanh u) / 2 is 1 / (1 + exp(-2u)) = s, so a value is f * s with s = rcp(1 + exp2(z)) and z a cubic
// of f: nine instructions, two of them quarter rate, and nothing to select (exp2 gives 0 or infinity past its range, and
// rcp(infinity) is 0). Two of the nine take s to s - 1/2 and back: half of the reference's tanh u = 2 s - 1 and 1 + tanh u, rounded where it rounds
// them, so that values far below 0 lose the digits there that they lose in the reference. With the tanh written out it was 22: a 2048 x 512 x 2048 product with bias and GELU merged 12.3 us, 11.2 now (without the GELU 9.9); 4 M
// values 6.1 -> 5.3. -2 u log2(e): the constants of the reference's formula, multiplied out.
__device__ __forceinline__ float gelu_exponent(float f) { return f * fmaf(f * f, -0.102943237f, -2.30220820f); }

// powf(f, 3.0f) of the reference formula: the cube formed in double and rounded once is the
// correctly rounded result, which is what a libm powf returns for this exponent, at a
// fraction of the cost of a general powf.
__device__ __forceinline__ float cube(float f) {
  const double d = (double)f;
  return (float)(d * d * d);
}


// ElemwiseOp.geluApprox (Elemwise.swift:109-111) on a value of tensor type T held as float; the
// caller multiplies by the scale (1 without scales) and rounds to T, as the element-wise kernel does.
template <bool HALF> __device__ __forceinline__ float gelu_approx(float f) {
  if (HALF) return f * (0.5f + (__builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gelu_exponent(f))) - 0.5f));
  return 0.5f * f * (1.0f + safe_tanh(0.797884561f * (f + 0.044715f * cube(f))));
}

// ElemwiseOp.geluApproxGrad (Elemwise.swift:112-119). Two general powf and a tanhf per element bound it by the vector ALU
// (4 M fp16 values: 38.5 us; now 7.6, with a scale array read along): the cube is gelu_approx's, squares are products, and results
// that are rounded to fp16 use the hardware's exp2 and reciprocal. There (1 + tanh u) / 2 and (1 - tanh^2 u) come
// straight from the sigmoids of +-2u, e^-2u / (1 + e^-2u) and 1 / (1 + e^-2u), with no subtraction of values next to 1 (so the tails keep their
// digits).
template <bool HALF> __device__ __forceinline__ float gelu_approx_grad(float f) {
  const float slope = 0.107032224435345f * (f * f) + 0.797884561f;
  if (HALF) {
    const float e = __builtin_amdgcn_exp2f(gelu_exponent(f));
    const float up = __builtin_amdgcn_rcpf(1.0f + e), down = fminf(e, 0x1p100f) * up;   // (no infinity times zero)
    return 2.0f * f * (up * down) * slope + up;
  }
  const float tanh_term = tanhf(0.035677408145115f * cube(f) + 0.797884561f * f);
  return 0.5f * f * (1.0f - tanh_term * tanh_term) * slope + 0.5f * tanh_term + 0.5f;
}
