// block_q4_0 quantize / dequantize kernels for gfx950.
//
// A thread owns one block (quantize) or two neighbouring ones (16-bit dequantize; four
// to fp32 in large calls) of a K block row; the one-column dequantize kernel takes
// every other shape.
#include "convert_common.h"

namespace mcq4 {

// Reference rule, quantization.py:333-369, for a weight of dtype DT (fp32,
// fp16 or bf16).  The reference runs every step as a torch op on the weight's
// own dtype, so each step here is one fp32 IEEE operation (the file is
// compiled with -ffp-contract=off) followed by a rounding to DT: amax (exact),
// amax/7, x/d, +8, round half to even (rintf, exact in DT), clamp.  For fp16
// and bf16 the fp32 result rounded to DT equals the correctly rounded DT
// operation (fp32 carries more than 2p + 2 bits for both, so the double rounding
// is innocuous).  d is stored as fp16 (d.to(float16), quantization.py:352), one
// more rounding for bf16.
//
// Quotients come from one IEEE reciprocal per block (div_by, bit-equal to the
// division) and roundings to DT from the hardware: with a division per element the
// arithmetic was half the time again in large calls.  One column per thread,
// although the accesses are narrow: the arithmetic of a block is a serial chain,
// and two or four columns of it in one thread leave too few waves in flight.
// us on fresh inputs, division per element / this / four (fp32: two) columns per thread:
// bf16 4096x14336 56.7 / 29.7 / 35.6 (a copy of the bytes 29), 4096x4096 18.7 / 11.1 /
// 15.1, 32x4096 5.3 / 3.2 / 6.5; fp16 1024x1024 4.0 / 3.6 / 6.9; fp32 4096x2048 10.6 /
// 9.1 / 11.4.
template <int DT>
__global__ void __launch_bounds__(256)
quantize_ref_kernel(const void *__restrict__ W, int64_t ldw, int nb, int N,
                    uint8_t *__restrict__ out) {
#pragma clang fp contract(off)
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    const int kb = blockIdx.y;
    if (n >= N || kb >= nb) return;
    const int64_t base = (int64_t)kb * QK * ldw + n;
    float x[QK];
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < QK; ++j) {
        x[j] = load_dt(W, base + (int64_t)j * ldw, DT);
        amax = fmaxf(amax, fabsf(x[j]));
    }
    float d = round_hw<DT>(amax / 7.0f);
    d = (d > 0.0f) ? d : 1.0f;
    uint16_t *dst = (uint16_t *)(out + ((int64_t)kb * N + n) * BLOCK_BYTES);
    uint32_t h[8];
    auto codes = [&](auto fast) {
        const float y = 1.0f / d;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            h[i] = 0;
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                float t0 = div_by<decltype(fast)::value, DT>(x[4 * i + e], d, y);
                float t1 = div_by<decltype(fast)::value, DT>(x[4 * i + e + 1], d, y);
                round_hw2<DT>(t0, t1);
                t0 += 8.0f; t1 += 8.0f;
                round_hw2<DT>(t0, t1);
                h[i] |= code4(t0, 15.0f) << (4 * e) | code4(t1, 15.0f) << (4 * e + 4);
            }
        }
    };
    if (__all(div_by_fits(d))) codes(std::true_type{});
    else codes(std::false_type{});
    dst[0] = bitcast<uint16_t>(to_half_exact(d));
#pragma unroll
    for (int i = 0; i < 8; ++i) dst[1 + i] = (uint16_t)h[i];
}

// llama.cpp quantize_row_q4_0_ref rule in the same layout: d = max_signed / -8,
// id = 1/d (0 if d == 0), q = min(15, trunc(x*id + 8.5)).
__global__ void __launch_bounds__(256)
quantize_llama_kernel(const float *__restrict__ W, int64_t ldw, int nb, int N,
                      uint8_t *__restrict__ out) {
#pragma clang fp contract(off)
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    const int kb = blockIdx.y;
    if (n >= N || kb >= nb) return;
    const float *src = W + (int64_t)kb * QK * ldw + n;
    float x[QK];
    float amax = 0.0f, mx = 0.0f;
#pragma unroll
    for (int j = 0; j < QK; ++j) {
        x[j] = src[(int64_t)j * ldw];
        if (amax < fabsf(x[j])) { amax = fabsf(x[j]); mx = x[j]; }
    }
    const float d = mx / -8.0f;
    const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
    uint32_t q[QK];
#pragma unroll
    for (int j = 0; j < QK; ++j) {
        float t = x[j] * id;   // two roundings: this file is built with -ffp-contract=off
        t = t + 8.5f;
        int v = (int)__builtin_truncf(t);
        v = v < 0 ? 0 : v;  // x*id >= -8 keeps t >= 0.5; guards non-finite input
        q[j] = (uint32_t)(v < 15 ? v : 15);
    }
    uint16_t *dst = (uint16_t *)(out + ((int64_t)kb * N + n) * BLOCK_BYTES);
    dst[0] = bitcast<uint16_t>(to_half_exact(d));
#pragma unroll
    for (int i = 0; i < 8; ++i)
        dst[1 + i] = (uint16_t)(q[4 * i] | (q[4 * i + 1] << 4) | (q[4 * i + 2] << 8) |
                                (q[4 * i + 3] << 12));
}

// quantization.py:396-419: W = (q - 8) * d, exact in fp32; the fp16 and bf16
// variants round that exact product once (nearest even).
template <int DT>
__global__ void __launch_bounds__(256)
dequant_kernel(const uint8_t *__restrict__ blocks, int nb, int N, void *__restrict__ out,
               int64_t ldo) {
#pragma clang fp contract(off)
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    const int kb = blockIdx.y;
    if (n >= N || kb >= nb) return;
    const uint16_t *b = (const uint16_t *)(blocks + ((int64_t)kb * N + n) * BLOCK_BYTES);
    const float d = (float)bitcast<_Float16>(b[0]);
    const int64_t o0 = (int64_t)kb * QK * ldo + n;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t w = b[1 + i];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = (float)((int)((w >> (4 * e)) & 0xF) - 8) * d;
            const int64_t o = o0 + (int64_t)(4 * i + e) * ldo;
            if constexpr (DT == DT_F16) ((_Float16 *)out)[o] = to_half_exact(v);
            else store_dt(out, o, v, DT);
        }
    }
}

// C neighbouring columns of one K block per thread (N % C == 0, blocks aligned to 2 C
// bytes, rows to C elements): the 18 C block bytes in dwords (C = 4: pairs), every
// output row as one store.  fp16: the exact q - 8 times d in one multiply, the
// single rounding of the exact product; bf16: that product rounded from fp32,
// where it is exact; fp32: exact.
// Bound by the output's bytes.  16 bits: C = 2 everywhere (us on fresh blocks, one
// column / 2 / 4: fp16 4096x4096 9.8 / 8.5 / 12.0, 4096x14336 35.2 / 27.3 / 28.8, 1024x1024
// 3.6 / 2.9 / 3.3; with four, 4096 columns leave two workgroups a CU).  fp32:
// dequant_wide_f32 below.
template <int DT, int C>
__global__ void __launch_bounds__(256)
dequant_wide_kernel(const uint8_t *__restrict__ blocks, int nb, int N, void *__restrict__ out, int64_t ldo) {
#pragma clang fp contract(off)
    typedef uint32_t in_t __attribute__((ext_vector_type(C / 2)));
    const int n = (blockIdx.x * 256 + threadIdx.x) * C, kb = blockIdx.y;
    if (n >= N) return;
    const in_t *src = (const in_t *)(blocks + ((int64_t)kb * N + n) * BLOCK_BYTES);
    uint32_t raw[9 * C / 2];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const in_t v = src[i];
#pragma unroll
        for (int j = 0; j < C / 2; ++j) raw[C / 2 * i + j] = v[j];
    }
    auto half_at = [&](int c, int i) { return (raw[(9 * c + i) / 2] >> (16 * ((9 * c + i) & 1))) & 0xFFFFu; };   // 2-byte word i of column c
    const int64_t o0 = (int64_t)kb * QK * ldo + n;
    const half2_t o1024 = {(_Float16)1032.0f, (_Float16)1032.0f};
#pragma unroll
    for (int i = 0; i < 8; ++i) {                 // rows 4 i .. 4 i + 3
        half2_t q01[C], q23[C];                   // q - 8 of the rows' pairs, per column
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const uint32_t w = half_at(c, 1 + i);
            q01[c] = bitcast<half2_t>((w & 0xFu) | ((w & 0xF0u) << 12) | 0x64006400u) - o1024;
            q23[c] = bitcast<half2_t>(((w >> 8) & 0xFu) | ((w & 0xF000u) << 4) | 0x64006400u) - o1024;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t o = o0 + (int64_t)(4 * i + e) * ldo;
            if constexpr (DT == DT_F16) {
                typedef _Float16 out_t __attribute__((ext_vector_type(C)));
                out_t v;
#pragma unroll
                for (int c = 0; c < C; ++c) v[c] = (e < 2 ? q01[c][e] : q23[c][e - 2]) * bitcast<_Float16>((uint16_t)half_at(c, 0));
                *(out_t *)((_Float16 *)out + o) = v;
            } else {
                typedef float out_t __attribute__((ext_vector_type(C)));
                out_t v;
#pragma unroll
                for (int c = 0; c < C; ++c)
                    v[c] = (float)(e < 2 ? q01[c][e] : q23[c][e - 2]) * (float)bitcast<_Float16>((uint16_t)half_at(c, 0));
                if constexpr (DT == DT_F32) {
                    *(out_t *)((float *)out + o) = v;
                } else {
                    in_t u;
#pragma unroll
                    for (int j = 0; j < C / 2; ++j)
                        u[j] = bitcast<uint32_t>(__builtin_convertvector((float2_t{v[2 * j], v[2 * j + 1]}), bf16x2_t));
                    *(in_t *)((uint16_t *)out + o) = u;
                }
            }
        }
    }
}

}  // namespace mcq4

// ---- launchers (called from the C ABI layer) -------------------------------
namespace mcq4 {

hipError_t launch_quantize_typed(int w_dtype, const void *W, int64_t ldw, int nb, int N,
                                 uint8_t *out, hipStream_t s) {
    dim3 grid((N + 255) / 256, nb), block(256);
    if (w_dtype == DT_F16)
        hipLaunchKernelGGL(quantize_ref_kernel<DT_F16>, grid, block, 0, s, W, ldw, nb, N, out);
    else if (w_dtype == DT_BF16)
        hipLaunchKernelGGL(quantize_ref_kernel<DT_BF16>, grid, block, 0, s, W, ldw, nb, N, out);
    else
        hipLaunchKernelGGL(quantize_ref_kernel<DT_F32>, grid, block, 0, s, W, ldw, nb, N, out);
    return hipGetLastError();
}

hipError_t launch_quantize(bool llama_rule, const float *W, int64_t ldw, int nb, int N,
                           uint8_t *out, hipStream_t s) {
    if (!llama_rule) return launch_quantize_typed(DT_F32, W, ldw, nb, N, out, s);
    dim3 grid((N + 255) / 256, nb), block(256);
    hipLaunchKernelGGL(quantize_llama_kernel, grid, block, 0, s, W, ldw, nb, N, out);
    return hipGetLastError();
}

// fp32 out: four columns per thread above 8 M weights if the threads that a row leaves idle
// are at most a sixteenth of N, above 11 M if they are at most a third of those launched; one
// column otherwise.  us on fresh blocks, one / four, none idle: 4096x4096 17.0 / 13.4,
// 2048x8192 16.2 / 13.0, 14336x14336 180 / 180, 4096x2048 8.1 / 8.0, 1024x1024 2.9 / 3.8.
// A third and less: 6816x2312 18.8 / 13.0, 6816x4104 29.4 / 23.5, 14336x2056 30.9 / 24.1,
// 3200x6400 19.3 / 15.7, 14336x2304 29.0 / 28.6, the worst 4096x3088 10.9 / 12.5; below 11 M
// 3200x3336 9.7 / 10.4, 1600x5376 8.2 / 8.9, the worst 1600x4104 7.5 / 6.7.  More:
// 14336x1064 16.1 / 19.2.  Over 172 shapes of 4 M to 57 M weights the line's mean time is
// 0.5 % above the better kernel's; that of one column alone 7.2 %, of four alone 3.3 %.
// On blocks that the last-level cache still holds: 2.5, 1.2 and 5.1 % (8192x1536 10.0 / 11.4).
static bool dequant_wide_f32(int nb, int N) {
    const int64_t weights = (int64_t)nb * QK * N, launched = ((int64_t)N + 1023) / 1024 * 1024, idle = launched - N;
    return (weights > (int64_t)8 << 20 && 16 * idle <= N) || (weights > (int64_t)11 << 20 && 3 * idle <= launched);
}

template <int DT>
static hipError_t launch_dequant_t(const uint8_t *blocks, int nb, int N, void *out, int64_t ldo, hipStream_t s) {
    constexpr int C = DT == DT_F32 ? 4 : 2;
    const bool wide = N % C == 0 && ldo % C == 0 && (uintptr_t)blocks % (2 * C) == 0 && (uintptr_t)out % (DT == DT_F32 ? 16 : 4) == 0 &&
                      (DT != DT_F32 || dequant_wide_f32(nb, N));
    if (wide) hipLaunchKernelGGL((dequant_wide_kernel<DT, C>), dim3((N / C + 255) / 256, nb), dim3(256), 0, s, blocks, nb, N, out, ldo);
    else hipLaunchKernelGGL(dequant_kernel<DT>, dim3((N + 255) / 256, nb), dim3(256), 0, s, blocks, nb, N, out, ldo);
    return hipGetLastError();
}

hipError_t launch_dequant(const uint8_t *blocks, int nb, int N, void *out, int64_t ldo, int out_dt, hipStream_t s) {
    if (out_dt == DT_F16) return launch_dequant_t<DT_F16>(blocks, nb, N, out, ldo, s);
    if (out_dt == DT_BF16) return launch_dequant_t<DT_BF16>(blocks, nb, N, out, ldo, s);
    return launch_dequant_t<DT_F32>(blocks, nb, N, out, ldo, s);
}

}  // namespace mcq4

// ---- workspace counter area -------------------------------------------------
namespace mcq4 {

// Zero-fills `n16` 16-byte words (a kernel rather than hipMemsetAsync, so the
// call can sit in a captured HIP graph).
__global__ void __launch_bounds__(256) zero16_kernel(uint4_t *p, int64_t n16) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n16) p[i] = uint4_t{0u, 0u, 0u, 0u};
}

hipError_t launch_zero_counters(void *ws, hipStream_t s) {
    const int64_t n16 = (int64_t)COUNTER_BYTES / 16;
    hipLaunchKernelGGL(zero16_kernel, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, s, (uint4_t *)ws, n16);
    return hipGetLastError();
}

}  // namespace mcq4
