// Per-group INT4 quantize / dequantize kernels (exact rounding; compiled with
// -ffp-contract=off so no multiply-add is fused).
//
// quantize (quantization.py:49-92): one thread per (column, range of groups).
// For an even group size a range is one group: the group's rows start at an
// even row, so no packed byte is shared between threads.  For an odd group
// size one thread walks every group of its column.  Per group: pass 1 finds
// min/max, then scale = R(R(max - min) / 15) clamped to >= R(1e-8),
// zero = R(-min / scale), and pass 2 quantizes q = rne(R(R(w / scale) + zero))
// clamped to [0, 15] (NaN -> 0), where R rounds to the weight dtype (the
// reference runs each step as a torch op in that dtype).  Rows come in pairs:
// an even row's q waits in a register for the odd row, and the byte is stored
// once.  Loads and stores are coalesced across the threads (columns).
//
// The GPU-side quantizer quantize_to_int4 (native/quant_kernels.metal:634-686,
// binding core_mps.mm:4655-4700) is the same computation in fp32 with Metal's
// round() (half away from zero); `away` selects it.
//
// dequantize (quantization.py:139-151): one thread per packed byte:
// w = R_out(((float)q - zero) * scale) for its two rows.
#include <math.h>

#include "convert_common.h"

namespace mcq4 {

struct I4QuantArgs {
    const void *W;
    int w_dt;
    int64_t ldw, K, N, gs, G;
    int64_t gpt;               // groups per thread (1, or G for odd group sizes)
    int away;                  // 1: round half away from zero (Metal round()), 0: half to even
    uint8_t *packed;
    void *scales, *zeros;
};

__global__ void __launch_bounds__(256) i4_quantize_kernel(I4QuantArgs a) {
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (n >= a.N) return;
    const int dt = a.w_dt;
    const float clamp_min = round_dt(1e-8f, dt);
    const int64_t nranges = (a.G + a.gpt - 1) / a.gpt;
    for (int64_t r = blockIdx.y; r < nranges; r += gridDim.y) {
        uint32_t pending = 0;
        const int64_t g_end = r * a.gpt + a.gpt < a.G ? r * a.gpt + a.gpt : a.G;
        for (int64_t g = r * a.gpt; g < g_end; ++g) {
            const int64_t k0 = g * a.gs;
            const int64_t k1 = k0 + a.gs < a.K ? k0 + a.gs : a.K;
            float mn = INFINITY, mx = -INFINITY;
            for (int64_t k = k0; k < k1; ++k) {
                const float w = load_dt(a.W, k * a.ldw + n, dt);
                mn = fminf(mn, w);
                mx = fmaxf(mx, w);
            }
            float scale = round_dt(round_dt(mx - mn, dt) / 15.0f, dt);
            scale = fmaxf(scale, clamp_min);
            const float zero = round_dt(-mn / scale, dt);
            store_dt(a.scales, g * a.N + n, scale, dt);
            store_dt(a.zeros, g * a.N + n, zero, dt);
            for (int64_t k = k0; k < k1; ++k) {
                const float w = load_dt(a.W, k * a.ldw + n, dt);
                const float t = round_dt(round_dt(w / scale, dt) + zero, dt);
                // rintf: half to even; roundf: half away from zero; fmaxf/fminf
                // map NaN to the bound 0.
                const float r = a.away ? roundf(t) : rintf(t);
                const uint32_t q = (uint32_t)fminf(fmaxf(r, 0.0f), 15.0f);
                if ((k & 1) == 0) {
                    pending = q;
                } else {
                    a.packed[(k >> 1) * a.N + n] = (uint8_t)(pending | (q << 4));
                }
            }
        }
    }
}

struct I4DequantArgs {
    const uint8_t *packed;
    const void *scales, *zeros;
    int sz_dt, out_dt;
    int64_t Kh, N, gs, ldo;
    void *out;
};

__global__ void __launch_bounds__(256) i4_dequant_kernel(I4DequantArgs a) {
    const int64_t total = a.Kh * a.N;
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += stride) {
        const int64_t kp = i / a.N, n = i - kp * a.N;
        const uint32_t b = a.packed[i];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t k = 2 * kp + h;
            const int64_t g = k / a.gs;
            const float s = load_dt(a.scales, g * a.N + n, a.sz_dt);
            const float z = load_dt(a.zeros, g * a.N + n, a.sz_dt);
            const float q = (float)((b >> (4 * h)) & 0xFu);
            const float w = (q - z) * s;
            store_dt(a.out, k * a.ldo + n, w, a.out_dt);
        }
    }
}

// The wide quantizer: groups of SL RPT rows (32, 64 or 128), C neighbouring columns
// per thread (N % C == 0, rows aligned to C elements).  A workgroup is 64 column
// sets x SL row slices of one group (a wave per slice): the weight is read once,
// C elements per load, its extremes meet in LDS, and the codes come from the
// registers -- quotients from one IEEE reciprocal per group and column (div_by,
// bit-equal to the division).  Bound by the weight's bytes beside the arithmetic:
// 4096x14336 bf16, groups of 128, 51.8 us (about 250 with one column per thread, two
// passes and a division per element; a copy of the bytes moved takes 29).  Eight
// slices of 16 rows were slower (quantize + dequantize 91.8 against 85.5).
template <int DT, int C, int SL, int RPT, bool AWAY>
__global__ void __launch_bounds__(64 * SL) i4_quantize_wide_kernel(I4QuantArgs a) {
#pragma clang fp contract(off)
    constexpr int ES = DT == DT_F32 ? 4 : 2, DW = C * ES / 4;   // dwords per row piece
    typedef uint32_t vec_t __attribute__((ext_vector_type(DW)));
    __shared__ float ext[2][SL][64][C];
    const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
    const int64_t n = ((int64_t)blockIdx.x * 64 + lane) * C;
    const bool live = n < a.N;
    const int64_t nn = live ? n : 0;
    const float clamp_min = round_hw<DT>(1e-8f);
    for (int64_t g = blockIdx.y; g < a.G; g += gridDim.y) {
        const int64_t k0 = g * (SL * RPT) + slice * RPT;
        const int rows = (int)(a.K - k0 < RPT ? (a.K - k0 > 0 ? a.K - k0 : 0) : RPT);   // even
        vec_t raw[RPT];
        float mn[C], mx[C];
#pragma unroll
        for (int c = 0; c < C; ++c) { mn[c] = INFINITY; mx[c] = -INFINITY; }
        const uint8_t *src = (const uint8_t *)a.W + (k0 * a.ldw + nn) * ES;
#pragma unroll
        for (int j = 0; j < RPT; ++j)
            if (j < rows) raw[j] = *(const vec_t *)(src + (int64_t)j * a.ldw * ES);
#pragma unroll
        for (int j = 0; j < RPT; ++j)
            if (j < rows) {
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const float w = elem_f32<DT>(raw[j][c * ES / 4], c);
                    mn[c] = fminf(mn[c], w);
                    mx[c] = fmaxf(mx[c], w);
                }
            }
#pragma unroll
        for (int c = 0; c < C; ++c) { ext[0][slice][lane][c] = mn[c]; ext[1][slice][lane][c] = mx[c]; }
        __syncthreads();
        float scale[C], zero[C], y[C];
        bool fits = true;
#pragma unroll
        for (int c = 0; c < C; ++c) {
#pragma unroll
            for (int q = 0; q < SL; ++q) {
                mn[c] = fminf(mn[c], ext[0][q][lane][c]);
                mx[c] = fmaxf(mx[c], ext[1][q][lane][c]);
            }
            scale[c] = fmaxf(round_hw<DT>(round_hw<DT>(mx[c] - mn[c]) / 15.0f), clamp_min);
            zero[c] = round_hw<DT>(-mn[c] / scale[c]);
            y[c] = 1.0f / scale[c];
            fits = fits && div_by_fits(scale[c]);
        }
        __syncthreads();                          // ext is free for the next group
        if (live && slice == 0) {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                store_dt(a.scales, g * a.N + n + c, scale[c], DT);
                store_dt(a.zeros, g * a.N + n + c, zero[c], DT);
            }
        }
        auto body = [&](auto fast) {
#pragma unroll
            for (int j = 0; j < RPT; j += 2) {
                if (j >= rows) break;
                uint32_t b = 0;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    float t0 = div_by<decltype(fast)::value, DT>(elem_f32<DT>(raw[j][c * ES / 4], c), scale[c], y[c]);
                    float t1 = div_by<decltype(fast)::value, DT>(elem_f32<DT>(raw[j + 1][c * ES / 4], c), scale[c], y[c]);
                    round_hw2<DT>(t0, t1);
                    t0 += zero[c]; t1 += zero[c];
                    round_hw2<DT>(t0, t1);
                    // rint: half to even; round: half away from zero; NaN -> 0.
                    const uint32_t q0 = (uint32_t)fminf(fmaxf(AWAY ? roundf(t0) : rintf(t0), 0.0f), 15.0f);
                    const uint32_t q1 = (uint32_t)fminf(fmaxf(AWAY ? roundf(t1) : rintf(t1), 0.0f), 15.0f);
                    b |= (q0 | q1 << 4) << (8 * c);
                }
                uint8_t *dst = a.packed + ((k0 + j) >> 1) * a.N + n;
                if constexpr (C == 4) *(uint32_t *)dst = b;
                else *(uint16_t *)dst = (uint16_t)b;
            }
        };
        if (live) {
            if (__all(fits)) body(std::true_type{});
            else body(std::false_type{});
        }
    }
}

// The wide dequantizer: four columns and eight byte rows per thread (N % 4 == 0,
// group sizes that are multiples of 16, aligned pointers): one scale and zero load
// per 16 rows, 4-byte packed loads, every output row as one 8- or 16-byte store.
// 4096x14336 to fp16 32.7 us, what a copy of the bytes moved takes.  From 384 K
// weights on: below, 16 rows of four columns a thread leave most of the CUs idle (us on
// fresh codes, one byte per thread / this: fp32 1024x256 3.2 / 3.4, fp16 128x1024 3.0 / 3.3,
// 32x4096 3.1 / 3.4; 512x1024 3.7 / 3.4, 32x14336 3.6 / 3.5).
template <int SZ, int OUT>
__global__ void __launch_bounds__(256) i4_dequant_wide_kernel(I4DequantArgs a) {
#pragma clang fp contract(off)
    const int64_t n = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (n >= a.N) return;
    for (int64_t r = blockIdx.y; r * 8 < a.Kh; r += gridDim.y) {
        const int64_t kp0 = r * 8, g = 2 * kp0 / a.gs;
        const int rows = (int)(a.Kh - kp0 < 8 ? a.Kh - kp0 : 8);
        uint32_t b[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < rows) b[i] = *(const uint32_t *)(a.packed + (kp0 + i) * a.N + n);
        float s[4], z[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            s[c] = load_dt(a.scales, g * a.N + n + c, SZ);
            z[c] = load_dt(a.zeros, g * a.N + n + c, SZ);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (i >= rows) break;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float w[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) w[c] = ((float)((b[i] >> (8 * c + 4 * h)) & 0xFu) - z[c]) * s[c];
                const int64_t o = (2 * (kp0 + i) + h) * a.ldo + n;
                if constexpr (OUT == DT_F32) {
                    *(float4_t *)((float *)a.out + o) = float4_t{w[0], w[1], w[2], w[3]};
                } else if constexpr (OUT == DT_F16) {
                    *(half4_t *)((_Float16 *)a.out + o) =
                        half4_t{to_half_exact(w[0]), to_half_exact(w[1]), to_half_exact(w[2]), to_half_exact(w[3])};
                } else {
                    const uint32_t lo = bitcast<uint32_t>(__builtin_convertvector((float2_t{w[0], w[1]}), bf16x2_t));
                    const uint32_t hi = bitcast<uint32_t>(__builtin_convertvector((float2_t{w[2], w[3]}), bf16x2_t));
                    *(u32x2 *)((uint16_t *)a.out + o) = u32x2{lo, hi};
                }
            }
        }
    }
}

template <int DT, int C, int SL, int RPT>
static void launch_i4_quantize_wide_t(const I4QuantArgs &a, hipStream_t s) {
    const dim3 grid((unsigned)((a.N / C + 63) / 64), (unsigned)(a.G < 65535 ? a.G : 65535));
    if (a.away) {
        if constexpr (DT == DT_F32) hipLaunchKernelGGL((i4_quantize_wide_kernel<DT, C, SL, RPT, true>), grid, dim3(64 * SL), 0, s, a);
    } else {
        hipLaunchKernelGGL((i4_quantize_wide_kernel<DT, C, SL, RPT, false>), grid, dim3(64 * SL), 0, s, a);
    }
}
template <int DT, int C>
static bool launch_i4_quantize_wide(const I4QuantArgs &a, hipStream_t s) {
    const int64_t es = DT == DT_F32 ? 4 : 2;
    if (a.N % C || a.ldw % C || (uintptr_t)a.W % (C * es) || (uintptr_t)a.packed % C) return false;
    if (a.gs == 32) launch_i4_quantize_wide_t<DT, C, 4, 8>(a, s);
    else if (a.gs == 64) launch_i4_quantize_wide_t<DT, C, 4, 16>(a, s);
    else if (a.gs == 128) launch_i4_quantize_wide_t<DT, C, 4, 32>(a, s);
    else return false;
    return true;
}

hipError_t launch_i4_quantize(const void *W, int w_dt, int64_t ldw, int64_t K, int64_t N,
                              int64_t gs, uint8_t *packed, void *scales, void *zeros,
                              hipStream_t s, int away) {
    I4QuantArgs a;
    a.away = away;
    a.W = W; a.w_dt = w_dt; a.ldw = ldw; a.K = K; a.N = N; a.gs = gs;
    a.G = (K + gs - 1) / gs;
    a.gpt = gs % 2 == 0 ? 1 : a.G;
    a.packed = packed; a.scales = scales; a.zeros = zeros;
    if (w_dt == DT_F16    ? launch_i4_quantize_wide<DT_F16, 4>(a, s)
        : w_dt == DT_BF16 ? launch_i4_quantize_wide<DT_BF16, 4>(a, s)
                          : launch_i4_quantize_wide<DT_F32, 2>(a, s))
        return hipGetLastError();
    const int64_t nranges = (a.G + a.gpt - 1) / a.gpt;
    const dim3 grid((unsigned)((N + 255) / 256), (unsigned)(nranges < 65535 ? nranges : 65535));
    hipLaunchKernelGGL(i4_quantize_kernel, grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_i4_dequant(const uint8_t *packed, const void *scales, const void *zeros,
                             int sz_dt, int64_t K, int64_t N, int64_t gs, void *out,
                             int64_t ldo, int out_dt, hipStream_t s) {
    I4DequantArgs a;
    a.packed = packed; a.scales = scales; a.zeros = zeros;
    a.sz_dt = sz_dt; a.out_dt = out_dt;
    a.Kh = K / 2; a.N = N; a.gs = gs; a.ldo = ldo; a.out = out;
    if (K * N >= 3 << 17 && N % 4 == 0 && ldo % 4 == 0 && gs % 16 == 0 && (uintptr_t)packed % 4 == 0 && (uintptr_t)out % (out_dt == DT_F32 ? 16 : 8) == 0) {
        const int64_t ry = (a.Kh + 7) / 8;
        const dim3 grid((unsigned)((N / 4 + 255) / 256), (unsigned)(ry < 65535 ? ry : 65535));
        auto go = [&](auto sz) {
            constexpr int SZ = decltype(sz)::value;
            if (out_dt == DT_F16) hipLaunchKernelGGL((i4_dequant_wide_kernel<SZ, DT_F16>), grid, dim3(256), 0, s, a);
            else if (out_dt == DT_BF16) hipLaunchKernelGGL((i4_dequant_wide_kernel<SZ, DT_BF16>), grid, dim3(256), 0, s, a);
            else hipLaunchKernelGGL((i4_dequant_wide_kernel<SZ, DT_F32>), grid, dim3(256), 0, s, a);
        };
        if (sz_dt == DT_F16) go(std::integral_constant<int, DT_F16>{});
        else if (sz_dt == DT_BF16) go(std::integral_constant<int, DT_BF16>{});
        else go(std::integral_constant<int, DT_F32>{});
        return hipGetLastError();
    }
    const int64_t total = a.Kh * N;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(i4_dequant_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace mcq4
