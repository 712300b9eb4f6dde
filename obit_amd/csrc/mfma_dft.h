// mfma_dft.h -- the parts the matrix-core DFT kernels share (dft.hip,
// beam.hip): phasors from FP64 phases, exchange between half-waves, FP16
// operand parts.
#pragma once
#include <hip/hip_runtime.h>
#include "phasor.h"

namespace obit {

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// e(t) for a phase in turns formed in FP64: reduced to [-1/2, 1/2] first,
// then the hardware sin / cos (HW) or the Taylor polynomial
template <bool HW>
__device__ __forceinline__ float2 eturn(double t) {
  float sn, cs;
  if (HW) sincos_turns_hw((float)(t - rint(t)), &sn, &cs);
  else sincos_turns_poly((float)(t - rint(t)), &sn, &cs);
  return make_float2(cs, sn);
}

// a value of the first half-wave (lanes 0..31) and of the second
// (32..63) in every lane: lo[l] = x[l mod 32], hi[l] = x[32 + l mod 32]
// (v_permlane32_swap exchanges lanes 32..63 of its first operand with
// lanes 0..31 of its second)
__device__ __forceinline__ void swap_halves(float2 x, float2 &lo, float2 &hi) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x.x), __float_as_uint(x.x), false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x.y), __float_as_uint(x.y), false, false);
  lo = make_float2(__uint_as_float(a[0]), __uint_as_float(b[0]));
  hi = make_float2(__uint_as_float(a[1]), __uint_as_float(b[1]));
}

// FP16 parts of (x, y), each pair packed in a 32-bit word (x in the low
// half): hi = fp16(x), fp16(y) rounded to nearest; lo = fp16(x - hi.x),
// fp16(y - hi.y), the differences formed in FP32 from the FP16 values.
// The differences are formed by v_fma_mix_f32 and packed by one conversion:
// v_fma_mixlo_f16 / v_fma_mixhi_f16, which would form and pack them in two
// instructions, issue at half rate (9 cycles measured against 5), so four
// full-rate instructions take fewer cycles than those three.
__device__ __forceinline__ void split_pair(float x, float y, unsigned &hi, unsigned &lo) {
  float dx, dy;
  asm("v_cvt_pk_f16_f32 %0, %4, %5\n\t"
      "v_fma_mix_f32 %2, -%0, 1.0, %4 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mix_f32 %3, -%0, 1.0, %5 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_cvt_pk_f16_f32 %1, %2, %3"
      : "=&v"(hi), "=&v"(lo), "=&v"(dx), "=&v"(dy)
      : "v"(x), "v"(y));
}

// (x, y) -> (y, -x) of an FP16 pair
__device__ __forceinline__ unsigned swap_neg(unsigned v) {
  unsigned r;
  asm("v_pk_add_f16 %0, %1, 0 op_sel:[1,0] op_sel_hi:[0,0] neg_hi:[1,0]" : "=v"(r) : "v"(v));
  return r;
}

}  // namespace obit
