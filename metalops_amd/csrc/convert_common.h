// Shared parts of the conversion kernels (q4_quant.hip, i4_convert.hip): exact
// division by a value shared by many elements, rounding to a dtype in hardware,
// packed element access.  The files are compiled with -ffp-contract=off.
#pragma once

#include <type_traits>

#include "q4_prefill.h"

namespace mcq4 {

// Rounds an fp32 value to fp16 (nearest even) with its sign of zero intact.
// The empty asm keeps the compiler from folding the preceding fp32 multiply and
// this conversion into v_fma_mix*_f16 with a +0 addend, which turns -0 into +0.
__device__ __forceinline__ _Float16 to_half_exact(float v) {
    asm volatile("" : "+v"(v));
    return (_Float16)v;
}

// x / d rounded to nearest even, with y = 1 / d rounded to nearest even.
// FAST (div_by_fits(d)): x y is within two ulps of the quotient; one residual step
// brings that below one ulp, and a second one from there is correctly rounded
// (Markstein, "Computation of elementary functions on the IBM RISC System/6000
// processor", 1990: q + (x - q d) y with q within one ulp and y correctly rounded,
// no underflow in the residual).  5 operations against the division's dozen.
// For 16-bit x and d, rounded to 16 bits next, one step does: a quotient of two
// p-bit values that is not itself a midpoint of p bits is at least 2^-(2p+1) of its
// size away from one (p = 11: 2^-23), twice the step's error, and a quotient that
// fp32 holds comes out exact.
// A residual can underflow only for quotients far below 2^-40, which no caller
// tells from zero.
template <bool FAST, int DT>
__device__ __forceinline__ float div_by(float x, float d, float y) {
    if constexpr (!FAST) return x / d;
    float q = x * y;
    q = __builtin_fmaf(__builtin_fmaf(-q, d, x), y, q);
    if constexpr (DT == DT_F32) q = __builtin_fmaf(__builtin_fmaf(-q, d, x), y, q);
    return q;
}
__device__ __forceinline__ bool div_by_fits(float d) { return d > 0x1p-60f && d < 0x1p60f; }

// round_dt in hardware (NaN stays NaN).
template <int DT>
__device__ __forceinline__ float round_hw(float x) {
    if constexpr (DT == DT_BF16) return (float)(__bf16)x;
    else if constexpr (DT == DT_F16) return (float)(_Float16)x;
    else return x;
}
template <int DT>
__device__ __forceinline__ void round_hw2(float &a, float &b) {
    if constexpr (DT == DT_BF16) {
        const uint32_t p = bitcast<uint32_t>(__builtin_convertvector((float2_t{a, b}), bf16x2_t));
        a = __uint_as_float(p << 16);
        b = __uint_as_float(p & 0xFFFF0000u);
    } else if constexpr (DT == DT_F16) {
        a = (float)(_Float16)a;
        b = (float)(_Float16)b;
    }
}

// Element c of a packed row piece, whose dword holding it is `w`, in fp32.
template <int DT>
__device__ __forceinline__ float elem_f32(uint32_t w, int c) {
    if constexpr (DT == DT_F32) return __uint_as_float(w);
    else if constexpr (DT == DT_BF16) return __uint_as_float((c & 1) ? w & 0xFFFF0000u : w << 16);
    else return (float)bitcast<_Float16>((uint16_t)((c & 1) ? w >> 16 : w));
}

// A code: t rounded half to even and clamped to [0, top] (NaN -> 0).
__device__ __forceinline__ uint32_t code4(float t, float top) {
    return (uint32_t)__builtin_rintf(fminf(fmaxf(t, 0.0f), top));
}

}  // namespace mcq4
