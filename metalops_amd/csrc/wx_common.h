// Shared parts of the any-activation matmul kernels (wx_gemm, wx_skinny):
// quantized weights (block_q4_0, per-group INT4, per-group INT8) times fp16, bf16
// or fp32 activations, any column count (INT4, INT8: 16 or more, groups of whole K
// steps), any 2-byte (q4_0) or byte (INT4, INT8) alignment of the weights.
//
// Semantics (quantization.py:207-239, :268-286, :452-454): the weight is
// dequantized in fp32 and rounded once to the activations' dtype, then
// Y = X @ W with fp32 sums and one rounding to the activations' dtype.
//
// Lane layout of a K step of 32 (MFMA 32x32): lane l supplies column (or row)
// l % 32 and the 16 K elements 16 (l / 32) .. +15 of the step.  The MFMA K order
// is a permutation of the real one, the same for both operands, so a lane's
// weights are contiguous: 8 nibble bytes of a q4_0 block, 8 byte rows of INT4,
// 16 of INT8.
#pragma once

#include <type_traits>

#include "q4_prefill.h"

namespace mcq4 {

enum : int { WX_Q4 = 0, WX_I4 = 1, WX_I8 = 2 };

struct WxArgs {
    const void *X;
    int64_t ldx;
    const uint8_t *W;            // q4_0 blocks, packed INT4 or int8 rows
    const void *scales, *zeros;  // INT4, INT8
    int sz_dt;
    void *Y;
    int64_t ldy;
    int M, K, N;
    // Group of K step k = mulhi(k, spg_mul) + (k & spg_one): spg_mul = ceil(2^32 / K
    // steps per group), or 0 with one group or one step per group (spg_one = ~0).
    uint32_t spg_mul, spg_one;
    int act;                     // ACT_*
    int S;                       // K splits (grid.z)
    float *part;                 // [S][M][ldp] fp32 partials when S > 1
    int ldp;
    int tiles_m, tiles_n;
    // wx_mid with S > 1: [column tiles][S] flag words behind the partials (null: the
    // reduction kernel sums), polls of a flag, splits treated as run on another XCD.
    uint32_t *flags = nullptr;
    uint32_t spin = 0, foreign = 0;
};

// Unaligned loads: gfx950 global loads need no alignment beyond the byte.
template <typename T>
__device__ __forceinline__ T load_u(const void *p) {
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

__device__ __forceinline__ float ubyte_f32(uint32_t v, int b) { return (float)((v >> (8 * b)) & 0xFFu); }

// Two fp32 values rounded (nearest even) to a pair of 16-bit activations' dtype.
template <int XT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (XT == DT_BF16) {
        return bitcast<uint32_t>(__builtin_convertvector((float2_t{a, b}), bf16x2_t));
    } else {
        return bitcast<uint32_t>(half2_t{(_Float16)a, (_Float16)b});
    }
}

// What a lane holds of the weights for one K step and TN column tiles: in flight
// (WxFly) and ready for wx_values (WxRaw).  q4_0: the same.  INT4 and INT8: a
// wave's 64 columns of a step's 16 (32) byte rows come as one (two) 16-byte loads
// per lane, four lanes on one row, and go through a wave's own LDS scratch to the
// lanes that own the columns (taken there directly, a row at a time, they are 8
// (16) loads of two bytes).
template <int WT, int TN>
struct WxRaw;
template <int TN>
struct WxRaw<WX_Q4, TN> {
    uint32_t q[TN][2];
    uint16_t d[TN];
};
template <int TN>
struct WxRaw<WX_I4, TN> {
    uint32_t q[8];               // byte rows, TN columns each
    uint32_t s[TN], z[TN];       // raw scale and zero (16 or 32 bits)
};
template <int TN>
struct WxRaw<WX_I8, TN> {
    uint32_t q[16];
    uint32_t s[TN], z[TN];
};
template <int WT, int TN>
struct WxFly {
    static_assert(TN == 2, "64 columns per wave");
    uint4_t v[WT == WX_I4 ? 1 : 2];
    uint32_t s[TN], z[TN];
};
template <int TN>
struct WxFly<WX_Q4, TN> : WxRaw<WX_Q4, TN> {};

// LDS scratch per wave: the step's rows of 64 bytes, the upper half of them (the
// lanes l / 32 = 1 read it) 64 bytes further on, on other banks.
constexpr int wx_scratch(int wt) { return wt == WX_Q4 ? 0 : (wt == WX_I4 ? 1024 : 2048) + 64; }

// The lane's place in the weights: its columns and the address of K step 0.
// q4_0: tile j's column is n0 + 32 j + l % 32.  INT4 and INT8: p = 2 (l % 32) + j of the
// wave's 64, in chunks of 16 columns that end at N at the latest (a chunk that
// would not is moved back: its columns are computed twice, with equal results).
template <int WT, int TN>
struct WxLane {
    int n[TN];
    int n0;                               // the workgroup-uniform column the offsets count from
    uint32_t off[WT == WX_Q4 ? TN : 1];   // byte offset in the step's rows
};
template <int WT, int TN>
__device__ __forceinline__ WxLane<WT, TN> wx_lane(const WxArgs &a, int n0, int lane) {
    WxLane<WT, TN> L;
    const int c = lane & 31;
    if constexpr (WT == WX_Q4) {
        L.n0 = min(n0, a.N - 1);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            L.n[j] = min(n0 + 32 * j + c, a.N - 1);
            L.off[j] = (uint32_t)(L.n[j] - L.n0) * BLOCK_BYTES;
        }
    } else {
        L.n0 = min(n0, a.N - 16);
#pragma unroll
        for (int j = 0; j < TN; ++j) L.n[j] = min(n0 + 16 * (c >> 3), a.N - 16) + ((2 * c + j) & 15);
        L.off[0] = (uint32_t)(lane >> 2) * (uint32_t)a.N + (uint32_t)(min(n0 + 16 * (lane & 3), a.N - 16) - L.n0);
    }
    return L;
}

template <int TN, bool SZ32>
__device__ __forceinline__ void wx_load_sz(const void *p, int64_t row, int n, uint32_t (&out)[TN]) {
    if constexpr (SZ32) {
        const u32x2 v = load_u<u32x2>((const float *)p + row + n);
        out[0] = v[0]; out[1] = v[1];
    } else {
        const uint32_t v = load_u<uint32_t>((const uint16_t *)p + row + n);
        out[0] = v & 0xFFFFu; out[1] = v >> 16;
    }
}

// Group of K step k: exact for k and steps per group below 2^16 (wx_supported).
__device__ __forceinline__ int wx_group(const WxArgs &a, int k) {
    return (int)(__umulhi((uint32_t)k, a.spg_mul) + ((uint32_t)k & a.spg_one));
}

// Loads K step `kb`.  TAIL: rows past K are clamped to the last one (wx_values
// zeroes their weights).
template <int WT, int TN, bool SZ32, bool TAIL>
__device__ __forceinline__ void wx_load(WxFly<WT, TN> &r, const WxArgs &a, const WxLane<WT, TN> &L, int kb, int lane) {
    if constexpr (WT == WX_Q4) {
        const uint8_t *base = a.W + ((int64_t)kb * a.N + L.n0) * BLOCK_BYTES;
        const int hi = lane >> 5;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint8_t *p = base + L.off[j];
            r.d[j] = load_u<uint16_t>(p);
            const u32x2 v = load_u<u32x2>(p + 2 + 8 * hi);
            r.q[j][0] = v[0]; r.q[j][1] = v[1];
        }
    } else {
        constexpr int LD = WT == WX_I4 ? 1 : 2;
        const uint8_t *base = a.W + (int64_t)kb * (16 * LD) * a.N + L.n0;
#pragma unroll
        for (int h = 0; h < LD; ++h) {
            const uint8_t *p = base + (int64_t)(16 * h) * a.N + L.off[0];
            if constexpr (TAIL) {                // back from row 16 h + lane / 4 to the last valid one
                const int over = kb * 16 * LD + 16 * h + (lane >> 2) - ((WT == WX_I4 ? a.K / 2 : a.K) - 1);
                p -= (int64_t)max(over, 0) * a.N;
            }
            r.v[h] = load_u<uint4_t>(p);
        }
        const int64_t row = (int64_t)wx_group(a, kb) * a.N;
        wx_load_sz<TN, SZ32>(a.scales, row, L.n[0], r.s);
        wx_load_sz<TN, SZ32>(a.zeros, row, L.n[0], r.z);
    }
}

// Orders a wave's LDS accesses before and after it, which other lanes of the wave make to the
// same bytes: without it only the lane's own addresses keep the compiler from moving one over
// the other.  The LDS runs a wave's accesses in order, so this is no instruction.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// A step's weights from flight to the lanes of their columns.  What keeps the compiler from
// moving the loads over the stores of their step or the next: the fence (FENCE), or a load
// address that it can't see through, so that each load may be to the bytes of any store.
// Against code with neither: the fence costs wx_skinny nothing (class means within 0.1 %)
// and wx_gemm up to 2.5 % (INT4 bf16 1755x1632x5248 74.3 -> 76.2 us), since it holds back the
// kernel's other LDS work too; the address leaves wx_gemm's class means at 0.992 to 1.001
// (that call 73.1 -> 73.3, most INT8 fp16 calls up to 3 % faster, the worst 300x4100x1025
// 44.1 -> 45.0) and costs wx_skinny up to 3.4 % (INT4 fp16 2x4100x14336 46.4 -> 48.0).
template <int WT, int TN, bool FENCE>
__device__ __forceinline__ WxRaw<WT, TN> wx_ready(const WxFly<WT, TN> &f, uint8_t *scratch, int lane) {
    if constexpr (WT == WX_Q4) {
        return f;
    } else {
        WxRaw<WT, TN> r;
        const int lrow = lane & 31, hi = lane >> 5;
        constexpr int HALF = WT == WX_I4 ? 512 + 64 : 1024 + 64, ROWS = WT == WX_I4 ? 8 : 16;
        uint32_t in_addr = lds_addr(scratch) + (uint32_t)(hi * HALF + 2 * lrow);
        if constexpr (!FENCE) asm("" : "+v"(in_addr));   // not volatile: one value for all steps
        const lds_u8 *const in = lds_ptr(in_addr);
        if constexpr (WT == WX_I4) {
            *(uint4_t *)(scratch + 16 * lane + 64 * hi) = f.v[0];
        } else {
            *(uint4_t *)(scratch + 16 * lane) = f.v[0];
            *(uint4_t *)(scratch + 1024 + 64 + 16 * lane) = f.v[1];
        }
        if constexpr (FENCE) wave_lds_order();
#pragma unroll
        for (int i = 0; i < ROWS; ++i) r.q[i] = *(const lds_u16 *)(in + 64 * i);
        if constexpr (FENCE) wave_lds_order();           // the next step stores to the same scratch
#pragma unroll
        for (int j = 0; j < TN; ++j) { r.s[j] = f.s[j]; r.z[j] = f.z[j]; }
        return r;
    }
}

// Both 16-bit readings and a select: a branch here would end the block that the
// loads and MFMAs around it are scheduled in.
template <bool SZ32>
__device__ __forceinline__ float wx_sz_f32(uint32_t v, int dt) {
    if constexpr (SZ32) return __uint_as_float(v);
    const float h = (float)bitcast<_Float16>((uint16_t)v), b = __uint_as_float(v << 16);
    return dt == DT_F16 ? h : b;
}

// q4_0 weights come out of a dword of nibbles (elements e0..e7) in the pair order
// [e0, e4, e1, e5, e2, e6, e3, e7]: two masks on the dword and on the dword
// shifted by 8, no byte moves.  wx_order puts 16-bit activations in that order
// (INT4 and INT8 keep the natural one); wx_slot is the element of slot s.
template <int WT>
__device__ __forceinline__ uint4_t wx_order(uint4_t x) {
    if constexpr (WT == WX_Q4)
        return uint4_t{__builtin_amdgcn_perm(x[2], x[0], 0x05040100u), __builtin_amdgcn_perm(x[2], x[0], 0x07060302u),
                       __builtin_amdgcn_perm(x[3], x[1], 0x05040100u), __builtin_amdgcn_perm(x[3], x[1], 0x07060302u)};
    else
        return x;
}
template <int WT>
constexpr int wx_slot(int s) {
    return WT == WX_Q4 ? (s & ~7) + ((s & 7) >> 1) + 4 * (s & 1) : s;
}

// The fp16 pairs {1024 + e0, 1024 + e4}, {64 + e1, 64 + e5}, ... of a nibble dword, exact.
__device__ __forceinline__ void q4_pairs(uint32_t w, uint32_t (&p)[4]) {
    const uint32_t mlo = opaque_sgpr(0x000F000Fu), mhi = opaque_sgpr(0x00F000F0u);
    const uint32_t e1024 = opaque_vgpr(0x64006400u), e64 = opaque_vgpr(0x54005400u);
    p[0] = and_or(w, mlo, e1024);
    p[1] = and_or(w, mhi, e64);
    p[2] = and_or(w >> 8, mlo, e1024);
    p[3] = and_or(w >> 8, mhi, e64);
}

// Whether a lane's block scale is infinite or NaN.
__device__ __forceinline__ bool q4_scale_odd(uint16_t d) { return (d & 0x7C00u) == 0x7C00u; }

// The eight weights of a nibble dword in fp32, in slot order.  FIN (d finite):
// (1024 + q) d - 1032 d and (64 + q) d - 72 d, one mixed-precision fma each, exact
// in fp32 (d has 11 significant bits).  Otherwise q - 8 first, so an infinite d
// gives the signed infinities of (q - 8) d.
template <bool FIN>
__device__ __forceinline__ void q4_values8(uint32_t q, float d, float *w) {
    const float c[2] = {-1032.0f * d, -72.0f * d};
    uint32_t p[4];
    q4_pairs(q, p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        half2_t v = bitcast<half2_t>(p[i]);
        if constexpr (!FIN) v -= (i & 1) ? half2_t{(_Float16)72.0f, (_Float16)72.0f} : half2_t{(_Float16)1032.0f, (_Float16)1032.0f};
        w[2 * i] = __builtin_fmaf((float)v[0], d, FIN ? c[i & 1] : 0.0f);
        w[2 * i + 1] = __builtin_fmaf((float)v[1], d, FIN ? c[i & 1] : 0.0f);
    }
}
// q - 8 of the eight in fp16, exact, in slot order.
__device__ __forceinline__ uint4_t q4_exact8(uint32_t q) {
    uint32_t p[4];
    q4_pairs(q, p);
    uint4_t r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const half2_t off = (i & 1) ? half2_t{(_Float16)72.0f, (_Float16)72.0f} : half2_t{(_Float16)1032.0f, (_Float16)1032.0f};
        r[i] = bitcast<uint32_t>(bitcast<half2_t>(p[i]) - off);
    }
    return r;
}
// The same eight as a B operand of 16-bit activations (fp16: one packed multiply,
// the single rounding of the exact product).
template <int XT, bool FIN>
__device__ __forceinline__ uint4_t q4_operand8(uint32_t q, uint16_t d) {
    uint4_t r;
    if constexpr (XT == DT_F16) {
#pragma clang fp contract(off)
        const uint32_t dd = d;
        const half2_t d2 = bitcast<half2_t>(dd | (dd << 16));
        uint32_t p[4];
        q4_pairs(q, p);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const half2_t off = (i & 1) ? half2_t{(_Float16)72.0f, (_Float16)72.0f} : half2_t{(_Float16)1032.0f, (_Float16)1032.0f};
            r[i] = bitcast<uint32_t>((bitcast<half2_t>(p[i]) - off) * d2);
        }
    } else {
        float w[8];
        q4_values8<FIN>(q, (float)bitcast<_Float16>(d), w);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = pack2<XT>(w[2 * i], w[2 * i + 1]);
    }
    return r;
}

// The lane's 16 weights of tile j in fp32, in slot order.  INT4 and INT8:
// (q - z) s in the reference's two fp32 roundings.
// TAIL: weights of rows past K are zero (`valid` = rows of the lane's 16 below K).
template <int WT, int XT, int TN, bool SZ32, bool TAIL, bool FIN>
__device__ __forceinline__ void wx_values(const WxRaw<WT, TN> &r, int j, int sz_dt, int valid, float (&w)[16]) {
    if constexpr (WT == WX_Q4) {
#pragma unroll
        for (int h = 0; h < 2; ++h) q4_values8<FIN>(r.q[j][h], (float)bitcast<_Float16>(r.d[j]), w + 8 * h);
    } else {
        const float s = wx_sz_f32<SZ32>(r.s[j], sz_dt), z = wx_sz_f32<SZ32>(r.z[j], sz_dt);
        auto val = [&](float q) {
#pragma clang fp contract(off)
            return (q - z) * s;
        };
        if constexpr (WT == WX_I4) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                w[2 * i] = val(ubyte_f32(r.q[i] & 0x0F0F0F0Fu, j));
                w[2 * i + 1] = val(ubyte_f32((r.q[i] >> 4) & 0x0F0F0F0Fu, j));
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) w[i] = val(ubyte_f32(r.q[i] ^ 0x80808080u, j) - 128.0f);
        }
        if constexpr (TAIL) {
#pragma unroll
            for (int i = 0; i < 16; ++i) w[i] = i < valid ? w[i] : 0.f;
        }
    }
}

// The B operands of tile j for 16-bit activations: ops[ks] = slots 8 ks .. +7 of
// the lane's 16.
template <int WT, int XT, int TN, bool SZ32, bool TAIL, bool FIN>
__device__ __forceinline__ void wx_operands(const WxRaw<WT, TN> &r, int j, int sz_dt, int valid, uint4_t (&ops)[2]) {
    if constexpr (WT == WX_Q4) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) ops[ks] = q4_operand8<XT, FIN>(r.q[j][ks], r.d[j]);
    } else {
        float w[16];
        wx_values<WT, XT, TN, SZ32, TAIL, FIN>(r, j, sz_dt, valid, w);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int u = 0; u < 4; ++u) ops[ks][u] = pack2<XT>(w[8 * ks + 2 * u], w[8 * ks + 2 * u + 1]);
    }
}

// body(FIN) with FIN = every lane's scales are finite (q4_0; always, otherwise).
template <int WT, int XT, int TN, typename F>
__device__ __forceinline__ void wx_if_finite(const uint16_t *d, F body) {
    if constexpr (WT == WX_Q4 && XT != DT_F16) {
        bool odd = false;
#pragma unroll
        for (int j = 0; j < TN; ++j) odd |= q4_scale_odd(d[j]);
        if (__builtin_expect(__any(odd), 0)) body(std::false_type{});
        else body(std::true_type{});
    } else {
        body(std::true_type{});
    }
}

template <int XT>
__device__ __forceinline__ float4_t wx_mfma16(uint4_t a, uint4_t b, float4_t c) {
    if constexpr (XT == DT_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<bf16x8_t>(a), bitcast<bf16x8_t>(b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<half8_t>(a), bitcast<half8_t>(b), c, 0, 0, 0);
}
template <int XT>
__device__ __forceinline__ float16_t wx_mfma(uint4_t a, uint4_t b, float16_t c) {
    return mfma32<XT>(bitcast<half8_t>(a), bitcast<half8_t>(b), c);
}

__device__ __forceinline__ float wx_activate(float y, int act) {
    if (act == ACT_SILU) return activate<ACT_SILU>(y);
    if (act == ACT_GELU) return activate<ACT_GELU>(y);
    return y;
}

// 16 bytes of activations (K elements k .. k + 16/ES - 1 of a row), any element
// alignment, zero past K.
template <int XT>
__device__ __forceinline__ uint4_t wx_load_x_any(const uint8_t *row, int k, int K) {
    uint4_t v = {0u, 0u, 0u, 0u};
    if constexpr (XT == DT_F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (k + e < K) v[e] = ((const uint32_t *)row)[k + e];
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (k + e < K) v[e / 2] |= (uint32_t)((const uint16_t *)row)[k + e] << (16 * (e & 1));
    }
    return v;
}

// ---- host ------------------------------------------------------------------
struct WxCall {
    int wt, x_dt, sz_dt, act;
    const void *X;
    int64_t ldx;
    const uint8_t *W;
    const void *scales, *zeros;
    void *Y;
    int64_t ldy;
    int64_t M, K, N, gs;
};
// Whether wx_gemm / wx_skinny take the call (any workspace, or none).
bool wx_supported(const WxCall &c);
size_t wx_workspace_bytes(int wt, int x_dt, int64_t M, int64_t K, int64_t N);
// ws may be null or too small: the plan then keeps K whole.
hipError_t launch_wx(const WxCall &c, void *ws, size_t ws_bytes, hipStream_t s);

}  // namespace mcq4
