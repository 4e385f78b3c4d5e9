// Any-activation decode and small-batch matmul, M <= 64 (wx_common.h): one
// 8-wave workgroup owns 32 TN columns; its waves split K, each a contiguous
// range of K steps, and sum through LDS in wave order.
//
//   * Weights and activations go from global memory straight into MFMA operand
//     registers, PF K steps ahead: no barrier until the end, any alignment.
//     Each weight is read and dequantized once.
//   * 32 TM activation rows (rows past M repeat the last one, their outputs are
//     not stored): the weights' bytes bound the kernel, not its MFMAs.
//   * fp32: a step's 32 products are summed from zero, then added (error as in wx_gemm).
//   * Split K over workgroups (grid.z) where the columns alone leave CUs idle:
//     fp32 partial rows summed in split order by wx_reduce_kernel.
//
// Bound by the latency of its loads (no LDS staging: a lane's 8 or 16 weight bytes and
// its row's activations per request) rather than by the bytes.  Sixteen waves instead of
// eight: slower (14.9 against 13.4 us).  Measured, against one thread per column with
// 2-byte weight loads: INT4 x bf16 M = 64 4096x14336 27.4 us (was 2472), INT4 x fp32 M =
// 32 4096x4096 19.8 (was 811).
#include <algorithm>
#include <type_traits>

#include "wx_common.h"

namespace mcq4 {

constexpr int WS_NW = 8, WS_TN = 2;

template <int WT, int XT, int TM, int TN, bool SZ32, bool ANY>
__global__ void __launch_bounds__(WS_NW * 64) wx_skinny_kernel(WxArgs a) {
    constexpr int ES = XT == DT_F32 ? 4 : 2;
    constexpr int XV = XT == DT_F32 ? 4 : 2;     // 16-byte activation loads per row tile and step
    // Ring slots: R - 1 K steps in flight beside the one in work.
    constexpr int R = TM == 2 && XT == DT_F32 ? 2 : 4;
    extern __shared__ __attribute__((aligned(16))) float red[];   // [waves][TM TN][16][64]; the loop: the waves' scratch
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 31, lhi = lane >> 5;
    const int n0 = blockIdx.x * (32 * TN), z = blockIdx.z;
    const int nks = (a.K + 31) / 32;
    const int ws = z * WS_NW + wave, wt = a.S * WS_NW;
    const int k_lo = (int)((int64_t)nks * ws / wt), nk = (int)((int64_t)nks * (ws + 1) / wt) - k_lo;

    const WxLane<WT, TN> L = wx_lane<WT, TN>(a, n0, lane);
    uint8_t *const scratch = (uint8_t *)red + wave * wx_scratch(WT);
    const uint8_t *xrow[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) xrow[i] = (const uint8_t *)a.X + (int64_t)min(32 * i + lrow, a.M - 1) * a.ldx * ES;

    struct Step {
        WxFly<WT, TN> r;
        uint4_t x[TM][XV];
    } ring[R];
    auto load = [&](Step &p, int kk) {
        const int kb = k_lo + min(kk, nk - 1);
        wx_load<WT, TN, SZ32, ANY && WT != WX_Q4>(p.r, a, L, kb, lane);
        const int k = kb * 32 + 16 * lhi;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int v = 0; v < XV; ++v) {
                if constexpr (ANY) p.x[i][v] = wx_load_x_any<XT>(xrow[i], k + v * (16 / ES), a.K);
                else p.x[i][v] = *(const uint4_t *)(xrow[i] + (int64_t)(k + v * (16 / ES)) * ES);
            }
    };

    std::conditional_t<XT == DT_F32, float[TM][TN][16], float16_t[TM][TN]> acc;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    auto step = [&](Step &p, int kk) {
        const int valid = a.K - (k_lo + kk) * 32 - 16 * lhi;
        if constexpr (XT != DT_F32) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) p.x[i][ks] = wx_order<WT>(p.x[i][ks]);
        }
        const WxRaw<WT, TN> raw = wx_ready<WT, TN, true>(p.r, scratch, lane);
        const uint16_t *d = nullptr;
        if constexpr (WT == WX_Q4) d = raw.d;
        wx_if_finite<WT, XT, TN>(d, [&](auto fin) {
            constexpr bool FIN = decltype(fin)::value;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (XT == DT_F32) {
                    float w[16];
                    float16_t part[TM];      // the step's 32 products, summed from zero
                    wx_values<WT, XT, TN, SZ32, ANY, FIN>(raw, j, a.sz_dt, valid, w);
#pragma unroll
                    for (int s = 0; s < 16; ++s) {
                        const int e = wx_slot<WT>(s);
#pragma unroll
                        for (int i = 0; i < TM; ++i)
                            part[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(p.x[i][e / 4][e % 4]), w[s],
                                                                           s ? part[i] : float16_t{}, 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            float v = acc[i][j][r] + part[i][r];
                            asm volatile("" : "+v"(v));   // else the add sinks to the next step, part with it
                            acc[i][j][r] = v;
                        }
                } else {
                    uint4_t B[2];
                    wx_operands<WT, XT, TN, SZ32, ANY, FIN>(raw, j, a.sz_dt, valid, B);
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                        for (int i = 0; i < TM; ++i) acc[i][j] = wx_mfma<XT>(p.x[i][ks], B[ks], acc[i][j]);
                }
            }
        });
    };

    if (nk > 0) {
        // The load of step k + R - 1 goes into the slot that step k - 1 has left, so no
        // value in flight is ever moved.
#pragma unroll
        for (int p = 0; p < R - 1; ++p) load(ring[p], p);
        for (int k0 = 0; k0 < nk; k0 += R) {
#pragma unroll
            for (int p = 0; p < R; ++p) {
                if (k0 + p >= nk) break;
                load(ring[(p + R - 1) % R], k0 + p + R - 1);
                __builtin_amdgcn_sched_barrier(0);
                step(ring[p], k0 + p);
            }
        }
    }

    if constexpr (WT != WX_Q4) __syncthreads();   // every wave is done with its scratch
    // Wave sums: lane l holds rows 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of each tile.
    constexpr int T = TM * TN;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (32 * i + 8 * (r >> 2) < a.M) red[((wave * T + i * TN + j) * 16 + r) * 64 + lane] = acc[i][j][r];
    __syncthreads();
#pragma unroll 1
    for (int v = tid; v < T * 1024; v += WS_NW * 64) {
        const int t = v >> 10, r = (v >> 6) & 15, i = t / TN, j = t % TN;
        const int m = 32 * i + 8 * (r >> 2) + 4 * lhi + (r & 3);
        const int c0 = n0 + (WT == WX_Q4 ? 32 * j + lrow : 16 * (lrow >> 3));
        if (m >= a.M || c0 >= a.N) continue;
        const int n = WT == WX_Q4 ? c0 : min(c0, a.N - 16) + ((2 * lrow + j) & 15);
        float sum = red[v];
#pragma unroll
        for (int w = 1; w < WS_NW; ++w) sum += red[w * T * 1024 + v];
        if (a.S > 1) a.part[((int64_t)z * a.M + m) * a.ldp + n] = sum;
        else store_dt(a.Y, (int64_t)m * a.ldy + n, wx_activate(sum, a.act), XT);
    }
}

hipError_t launch_wx_reduce(const WxArgs &a, int x_dt, hipStream_t s);
hipError_t launch_wx_gemv(const WxArgs &a, int x_dt, bool any, hipStream_t s);
bool wx_mid_shape(int wt, int x_dt, int64_t M, int64_t N);
bool wx_mid_supported(const WxCall &c);
int wx_mid_splits(int64_t K, int64_t N);
size_t wx_mid_flag_bytes(int64_t N, int S);
hipError_t launch_wx_mid(WxArgs a, int x_dt, bool *reduce, hipStream_t s);
hipError_t launch_wx_gemm(WxArgs a, int wt, int x_dt, bool any, hipStream_t s);
int wx_gemm_splits(int x_dt, int64_t M, int64_t K, int64_t N);

template <int WT, int XT, int TM, int TN, bool SZ32, bool ANY>
static hipError_t launch_wx_skinny_k(const WxArgs &a, hipStream_t s) {
    const size_t lds = (size_t)WS_NW * TM * TN * 1024 * sizeof(float);
    const dim3 grid((a.N + 32 * TN - 1) / (32 * TN), 1, a.S);
    if (lds > 64 * 1024)
        if (hipError_t e = hipFuncSetAttribute((const void *)wx_skinny_kernel<WT, XT, TM, TN, SZ32, ANY>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds))
            return e;
    hipLaunchKernelGGL((wx_skinny_kernel<WT, XT, TM, TN, SZ32, ANY>), grid, dim3(WS_NW * 64), lds, s, a);
    return hipGetLastError();
}
template <int WT, int XT, bool SZ32>
static hipError_t launch_wx_skinny_t(const WxArgs &a, bool any, hipStream_t s) {
    constexpr int TN = WS_TN;
    if (a.M <= 32)
        return any ? launch_wx_skinny_k<WT, XT, 1, TN, SZ32, true>(a, s) : launch_wx_skinny_k<WT, XT, 1, TN, SZ32, false>(a, s);
    return any ? launch_wx_skinny_k<WT, XT, 2, TN, SZ32, true>(a, s) : launch_wx_skinny_k<WT, XT, 2, TN, SZ32, false>(a, s);
}
template <int WT, bool SZ32>
static hipError_t launch_wx_skinny_s(const WxArgs &a, int x_dt, bool any, hipStream_t s) {
    if (x_dt == DT_F16) return launch_wx_skinny_t<WT, DT_F16, SZ32>(a, any, s);
    if (x_dt == DT_BF16) return launch_wx_skinny_t<WT, DT_BF16, SZ32>(a, any, s);
    return launch_wx_skinny_t<WT, DT_F32, SZ32>(a, any, s);
}
template <int WT>
static hipError_t launch_wx_skinny_w(const WxArgs &a, int x_dt, bool any, hipStream_t s) {
    if constexpr (WT != WX_Q4)
        if (a.sz_dt == DT_F32) return launch_wx_skinny_s<WT, true>(a, x_dt, any, s);
    return launch_wx_skinny_s<WT, false>(a, x_dt, any, s);
}

// K splits: one workgroup per CU, every wave at least 2 K steps.
static int wx_skinny_splits(int64_t K, int64_t N) {
    const int64_t t = (N + 32 * WS_TN - 1) / (32 * WS_TN), nks = (K + 31) / 32;
    int S = 1;
    while (t * S * 2 <= 256 && nks / (S * 2 * WS_NW) >= 2 && S < 16) S *= 2;
    return S;
}

static int64_t wx_ldp(int64_t N) { return (N + 3) / 4 * 4; }

// Partials of q4_0 x fp16 stay within 16 MiB, what the allocation-free entry point holds.
// q4_0 in 16 bits below K = 768 with 1 M outputs or more: no split, whose partials (16 bytes of
// traffic an output, at about 5 TB/s) and second launch cost more than half the K steps: us,
// two splits / none: 2048x512x1001 24.7 / 18.2, 300x512x6001 24.7 / 18.3, 128x640x14335 25.4 / 20.7.
static int wx_splits(int wt, int x_dt, int64_t M, int64_t K, int64_t N) {
    if (wt == WX_Q4 && M <= 16) return 1;         // wx_gemv
    // One plan for a shape, whatever the alignment: wx_mid and wx_skinny share it.
    int S = wx_mid_shape(wt, x_dt, M, N) ? wx_mid_splits(K, N) : M <= 64 ? wx_skinny_splits(K, N) : wx_gemm_splits(x_dt, M, K, N);
    if (wt == WX_Q4 && x_dt != DT_F32 && M > 64 && K < 768 && M * N >= (1 << 20)) S = 1;
    if (wt == WX_Q4 && x_dt == DT_F16)
        while (S > 1 && (int64_t)S * M * wx_ldp(N) * 4 > ((int64_t)16 << 20)) S /= 2;
    return S;
}

size_t wx_workspace_bytes(int wt, int x_dt, int64_t M, int64_t K, int64_t N) {
    const int S = wx_splits(wt, x_dt, M, K, N);
    // Partials follow the counter area, which other kernels rely on staying zero.
    if (S == 1) return 0;
    return COUNTER_BYTES + (size_t)S * M * wx_ldp(N) * sizeof(float) +
           (wx_mid_shape(wt, x_dt, M, N) ? wx_mid_flag_bytes(N, S) : 0);
}

// Every q4_0 call; INT4 and INT8 with groups of whole K steps, at least 16
// columns (a lane loads 16 at a time), 16 rows within a 32-bit offset and a
// K that keeps the group's multiply-high exact.  The fused
// activations exist for INT4 x fp16 only.
bool wx_supported(const WxCall &c) {
    if (c.wt != WX_Q4 && (c.gs % 32 != 0 || c.N < 16 || c.N > (1 << 27) || c.K > 65535 * 32)) return false;
    if (c.act != ACT_NONE && (c.wt != WX_I4 || c.x_dt != DT_F16)) return false;
    return true;
}

hipError_t launch_wx(const WxCall &c, void *ws, size_t ws_bytes, hipStream_t s) {
    WxArgs a;
    a.X = c.X; a.ldx = c.ldx; a.W = c.W; a.scales = c.scales; a.zeros = c.zeros; a.sz_dt = c.sz_dt;
    a.Y = c.Y; a.ldy = c.ldy; a.M = (int)c.M; a.K = (int)c.K; a.N = (int)c.N;
    const int64_t spg = c.wt == WX_Q4 ? 1 : c.gs / 32;
    a.spg_mul = spg * 32 >= c.K ? 0u : (uint32_t)((((uint64_t)1 << 32) + spg - 1) / spg);
    a.spg_one = 0u;
    if (spg == 1) { a.spg_mul = 0u; a.spg_one = ~0u; }   // 2^32 itself does not fit
    a.act = c.act;
    a.S = wx_splits(c.wt, c.x_dt, c.M, c.K, c.N);
    if (a.S > 1 && (!ws || ws_bytes < wx_workspace_bytes(c.wt, c.x_dt, c.M, c.K, c.N))) a.S = 1;
    a.ldp = (int)wx_ldp(c.N);
    a.part = a.S > 1 ? (float *)((char *)ws + COUNTER_BYTES) : nullptr;
    a.tiles_m = a.tiles_n = 0;
    const int es = c.x_dt == DT_F32 ? 4 : 2;
    const bool any = (uintptr_t)c.X % 16 != 0 || (c.ldx * es) % 16 != 0 || c.K % 32 != 0;
    if (c.wt == WX_Q4 && c.M <= 16) return launch_wx_gemv(a, c.x_dt, any, s);
    if (c.M > 64) return launch_wx_gemm(a, c.wt, c.x_dt, any, s);
    bool reduce = a.S > 1;
    const hipError_t e = wx_mid_supported(c) ? launch_wx_mid(a, c.x_dt, &reduce, s)
                         : c.wt == WX_Q4   ? launch_wx_skinny_w<WX_Q4>(a, c.x_dt, any, s)
                         : c.wt == WX_I4 ? launch_wx_skinny_w<WX_I4>(a, c.x_dt, any, s)
                                         : launch_wx_skinny_w<WX_I8>(a, c.x_dt, any, s);
    if (e != hipSuccess || !reduce) return e;
    return launch_wx_reduce(a, c.x_dt, s);
}

}  // namespace mcq4
