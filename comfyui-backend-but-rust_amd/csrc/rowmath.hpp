// The activation functions of the row prologues (csrc/common.cuh:71-95), shared by the prologue kernels and the quantizer.
// exp, expm1, erf and tanh are evaluated in fp64 and rounded to fp32, i.e. correctly rounded fp32 functions: the
// reference calls CUDA's expf / erff / tanhf, 1-2 ulp routines whose bits only a run could show.
#pragma once
#include "common.hpp"

// Kept out of line: the fp64 routines are long, and the callers evaluate them 16 times per lane in many kernel variants.
static __device__ __attribute__((noinline)) float exp_cr(float x) { return (float)exp((double)x); }
__device__ __forceinline__ float silu_f(float x) { return x / (1.f + exp_cr(-x)); }          // csrc/common.cuh:71
__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + exp_cr(-x)); }     // :72
static __device__ __attribute__((noinline)) float stable_tanh(float x) {                                      // :74-77
    const float t = (float)expm1((double)(-2.f * fabsf(x)));
    return copysignf(-t / (t + 2.f), x);
}
static __device__ __attribute__((noinline)) float gelu_f(float x) { return 0.5f * x * (1.f + (float)erf((double)(x * 0.70710678118654752f))); }  // :91
static __device__ __attribute__((noinline)) float gelu_tanh_f(float x) {                                      // :92-95
    const float k0 = 0.7978845608028654f, k1 = 0.044715f;
    return 0.5f * x * (1.f + (float)tanh((double)(k0 * __builtin_fmaf(k1 * x * x, x, x))));
}

// MOSS Image's soft-capped gated activation as one float expression, csrc/common.cuh:80-82:
//   4.f * stable_tanh(gate / 4.f) / (1.f + expf(-gate)) * (25.f * stable_tanh(hidden / 25.f))
// evaluated left to right: (gate factor) * (hidden factor), each an fp32 value of one argument.
__device__ __forceinline__ float situ_gate_f(float gate) { return 4.f * stable_tanh(gate / 4.f) / (1.f + exp_cr(-gate)); }
__device__ __forceinline__ float situ_hidden_f(float hidden) { return 25.f * stable_tanh(hidden / 25.f); }
__device__ __forceinline__ float situ_f(float hidden, float gate) { return situ_gate_f(gate) * situ_hidden_f(hidden); }

// sigmoid_f and silu_f, to be rounded to bf16, for a bf16 x, from the hardware's exp2 and reciprocal (one unit in the last
// place of fp32 each): every one of the 65536 inputs gives the bits that rounding the functions above gives (a GPU test
// goes through them all).  About 24 cycles of a SIMD per wave; a 128 KB table read per lane from global memory, as the
// other activations do, costs the CU's address path 64.  1 + e is scaled so that its reciprocal stays in the normal range
// up to the overflow of e, which gives 0 as dividing by an infinite fp32 does.  The scale's 9/8 is there because with a
// plain power of two one input, silu(5.9375), falls on the other side of a rounding boundary.
__device__ __forceinline__ float sigmoid_of_bf16(float x) {
    constexpr float c = 1.125f * 0x1p-32f;
    const float e = __builtin_amdgcn_exp2f(x * -1.44269504088896340736f);
    return __builtin_amdgcn_rcpf(__builtin_fmaf(e, c, c)) * c;
}
__device__ __forceinline__ float silu_of_bf16(float x) { return x * sigmoid_of_bf16(x); }
