// Shared plan and arguments of the LDS-staged q4_0 prefill GEMM (q4_gemm6):
// output tiles of 128 x 256, optional split-K over grid.z with fp32 partial
// tiles in the caller's workspace.
#pragma once

#include "i4_common.h"

namespace mcq4 {

constexpr int G6_BM = 128;   // output tile rows
constexpr int G6_BN = 256;   // output tile columns

// The prefill kernels take fp16 or bf16 activations (XT = DT_F16 / DT_BF16, 16
// bits either way; X and Y are addressed as _Float16): the MFMA, the weights'
// rounding and the store are of that dtype.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));

template <int XT>
__device__ __forceinline__ float16_t mfma32(half8_t a, half8_t b, float16_t c) {
    if constexpr (XT == DT_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(bitcast<bf16x8_t>(a), bitcast<bf16x8_t>(b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Second half of the dequant of two weights: `h` is the fp16 pair {1024 + q0, 64 + q1}
// (exact); minus {1032, 72} (exact) gives q - 8, and the product with d is
// rounded once to XT.  fp16: one packed multiply.  bf16: the exact products in
// fp32 (d has 11 significant bits), then one packed conversion.
template <int XT>
struct Q4Scale {
    half2_t d2;
    __device__ __forceinline__ void set(uint32_t dd) { d2 = bitcast<half2_t>(__builtin_amdgcn_perm(dd, dd, 0x01000100u)); }
    __device__ __forceinline__ uint32_t weights(uint32_t h) const {
#pragma clang fp contract(off)
        const half2_t off = {(_Float16)1032.0f, (_Float16)72.0f};
        return bitcast<uint32_t>((bitcast<half2_t>(h) - off) * d2);
    }
};
template <>
struct Q4Scale<DT_BF16> {
    uint32_t dd;
    __device__ __forceinline__ void set(uint32_t v) { dd = v; }
    __device__ __forceinline__ uint32_t weights(uint32_t h) const {
        const half2_t off = {(_Float16)1032.0f, (_Float16)72.0f};
        const half2_t p = bitcast<half2_t>(h) - off;
        const float d = (float)bitcast<_Float16>((uint16_t)dd);
        const float2_t w = {__builtin_fmaf((float)p[0], d, 0.0f), __builtin_fmaf((float)p[1], d, 0.0f)};
        return bitcast<uint32_t>(__builtin_convertvector(w, bf16x2_t));
    }
};

// fp32 rounded to XT, as the bits stored through a _Float16 pointer.
template <int XT>
__device__ __forceinline__ _Float16 out16(float v) {
    if constexpr (XT == DT_BF16) return bitcast<_Float16>((__bf16)v);
    else return (_Float16)v;
}

struct Gemm6Args {
    const _Float16 *X;
    int64_t ldx;
    const uint8_t *W;
    _Float16 *Y;
    int64_t ldy;
    int M, nb, N;
    int tiles_m, tiles_n;
    int S;               // K splits (grid.z)
    float *partials;     // [tiles][S][128*256] when S > 1
    // S == 2 with an XCD-local exchange: grid.x padded to a multiple of 8, the
    // second split of a tile to finish adds the first's partial and stores Y
    // (64-bit tickets [8][4096] by blockIdx.x mod 8 at the workspace start).
    uint64_t *tickets = nullptr;
    uint32_t foreign = 0;    // splits treated as run on another XCD (test switch)
};

// Needs N % 8 == 0, 16-byte aligned W and activation rows, K >= 32, M * ldx <
// 2^30 and W below 2^31 bytes (buffer loads).
bool gemm6_supported(const _Float16 *X, int64_t ldx, const uint8_t *W, int64_t M, int64_t K, int64_t N);
size_t gemm6_workspace_bytes(int64_t M, int64_t K, int64_t N);
hipError_t launch_gemm6(const _Float16 *X, int64_t ldx, const uint8_t *W, _Float16 *Y,
                        int64_t ldy, int M, int K, int N, int x_dt, void *ws, hipStream_t s);

// Few-tile prefill GEMM (q4_gemm8): 128 x 128 tiles, eight waves with K split
// four ways inside the workgroup, at most two K splits across workgroups
// summed through the XCD's L2 (partials [tiles][2][128*128] after the ticket
// area).  Needs what q4_gemm6 needs.
constexpr int G8_BM = 128;
constexpr int G8_BN = 128;
bool gemm8_supported(const _Float16 *X, int64_t ldx, const uint8_t *W, int64_t M, int64_t K, int64_t N);
size_t gemm8_workspace_bytes(int64_t M, int64_t K, int64_t N);
int gemm8_workgroups(int64_t M, int64_t K, int64_t N);   // tiles x K splits of its plan
hipError_t launch_gemm8(const _Float16 *X, int64_t ldx, const uint8_t *W, _Float16 *Y,
                        int64_t ldy, int M, int K, int N, int x_dt, void *ws, hipStream_t s);

}  // namespace mcq4
