// Any-activation prefill matmul (wx_common.h): 128 x 256 tiles, four waves of
// 128 x 64 (MFMA 32x32, 128 fp32 accumulators), two workgroups per CU.
//
//   * Weights go from global memory straight into registers, PF K steps of 32
//     ahead: a wave owns its 64 columns, so each weight is read and dequantized
//     once per workgroup, and no alignment beyond the format's own is needed
//     (any N, any row offset).
//   * Activations: one stage (128 bytes of each of the 128 rows: 64 K elements
//     in 16 bits, 32 in fp32) goes through registers into one of two LDS slots,
//     loaded a whole stage ahead; chunk c of row r sits at c ^ (r & 7), so the
//     16-byte operand reads are free of bank conflicts.  ANY: activations that
//     are not 16-byte aligned, or a K that is no multiple of 32, are read
//     element by element, zero past K.
//   * 16-bit activations: v_mfma_f32_32x32x16_{f16,bf16}, a B operand feeding
//     four MFMAs.  fp32: v_mfma_f32_32x32x2_f32, weights kept in fp32.
//   * Split K (grid.z) for outputs with few tiles: fp32 partial rows summed in
//     split order by wx_reduce_kernel.
//
// Replaces one-thread-per-column VALU kernels that re-read every weight for each
// 8 rows.  Measured: q4_0 x bf16 M = 512 4096x4096 66 us (258 TFLOP/s), was 2111;
// INT4 x bf16 M = 256 4096x11008 195 us, was 8180.
#include <algorithm>

#include "wx_common.h"

namespace mcq4 {

constexpr int WG_BM = 128, WG_BN = 256, WG_TM = 4, WG_TN = 2;
constexpr int WG_SLOT = WG_BM * 128;
#ifndef WX_PF_SET
constexpr int WG_PF = 2;                       // K steps of weights in flight
#else
constexpr int WG_PF = WX_PF_SET;
#endif

template <int WT, int XT, bool ANY, bool ACT>
__global__ void __launch_bounds__(256, 2) wx_gemm_kernel(WxArgs a) {
    constexpr int ES = XT == DT_F32 ? 4 : 2;
    constexpr int STEPS = XT == DT_F32 ? 1 : 2;  // K steps of 32 per stage
    __shared__ __attribute__((aligned(16))) uint8_t sA[2 * WG_SLOT];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 31, lhi = lane >> 5;

    const int bid = blockIdx.x, gx = gridDim.x;
    int tile_id = bid;
    if (gx % 8 == 0) tile_id = (bid % 8) * (gx / 8) + bid / 8;
    const int m0 = (tile_id % a.tiles_m) * WG_BM, n0 = (tile_id / a.tiles_m) * WG_BN + 64 * wave;
    const int nks = (a.K + 31) / 32;
    const int z = blockIdx.z;
    const int k_lo = (int)((int64_t)nks * z / a.S), nk = (int)((int64_t)nks * (z + 1) / a.S) - k_lo;

    const WxLane<WT, WG_TN> L = wx_lane<WT, WG_TN>(a, n0, lane);

    // Activation copies: thread t moves chunks (row (t + 256 u) / 8, chunk t % 8), u < 4.
    const uint8_t *xrow[4];
    const int xc = tid & 7;
#pragma unroll
    for (int u = 0; u < 4; ++u)
        xrow[u] = (const uint8_t *)a.X + (int64_t)min(m0 + (tid >> 3) + 32 * u, a.M - 1) * a.ldx * ES;
    uint4_t xs[4];
    auto load_a = [&](int st) {
        const int k = (k_lo + st * STEPS) * 32 + xc * (16 / ES);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if constexpr (ANY) {
                xs[u] = wx_load_x_any<XT>(xrow[u], k, a.K);
            } else {
                // Past the split's end (an odd last stage): any valid chunk, no MFMA uses it.
                xs[u] = *(const uint4_t *)(xrow[u] + (int64_t)min(k, a.K - 16 / ES) * ES);
            }
        }
    };
    auto store_a = [&](int slot) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int r = (tid >> 3) + 32 * u;
            *(uint4_t *)(sA + slot * WG_SLOT + r * 128 + ((xc ^ (r & 7)) << 4)) = xs[u];
        }
    };
    auto read_a = [&](int slot, int i, int chunk) {
        const int r = 32 * i + lrow;
        return *(const uint4_t *)(sA + slot * WG_SLOT + r * 128 + ((chunk ^ (lrow & 7)) << 4));
    };

    WxRaw<WT, WG_TN> raw[WG_PF];
    int kld = 0, grp = WT == WX_Q4 ? 0 : k_lo / a.spg, gcnt = WT == WX_Q4 ? 0 : k_lo % a.spg;
    auto load_w = [&](WxRaw<WT, WG_TN> &r) {
        wx_load<WT, WG_TN, ANY && WT != WX_Q4>(r, a, L, k_lo + kld, grp, lane);
        if (kld + 1 < nk) {                      // past the split's end: its last step again
            ++kld;
            if (WT != WX_Q4 && ++gcnt == a.spg) { gcnt = 0; ++grp; }
        }
    };

    float16_t acc[WG_TM][WG_TN];
#pragma unroll
    for (int i = 0; i < WG_TM; ++i)
#pragma unroll
        for (int j = 0; j < WG_TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    auto step = [&](int slot, int t, int kk, WxRaw<WT, WG_TN> &r) {
        const int valid = a.K - (k_lo + kk) * 32 - 16 * lhi;
        if constexpr (XT == DT_F32) {
            float w[WG_TN][16];
#pragma unroll
            for (int j = 0; j < WG_TN; ++j) wx_values<WT, XT, WG_TN, ANY>(r, j, a.sz_dt, valid, w[j]);
            load_w(r);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float4_t x[WG_TM];
#pragma unroll
                for (int i = 0; i < WG_TM; ++i) x[i] = bitcast<float4_t>(read_a(slot, i, 4 * lhi + q));
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < WG_TM; ++i)
#pragma unroll
                        for (int j = 0; j < WG_TN; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i][e], w[j][4 * q + e], acc[i][j], 0, 0, 0);
            }
        } else {
            uint4_t B[WG_TN][2];
#pragma unroll
            for (int j = 0; j < WG_TN; ++j) wx_operands<WT, XT, WG_TN, ANY>(r, j, a.sz_dt, valid, B[j]);
            load_w(r);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int i = 0; i < WG_TM; ++i) {
                    const uint4_t x = read_a(slot, i, 4 * t + 2 * lhi + ks);
#pragma unroll
                    for (int j = 0; j < WG_TN; ++j) acc[i][j] = wx_mfma<XT>(x, B[j][ks], acc[i][j]);
                }
        }
    };

    static_assert(WG_PF % STEPS == 0 || STEPS == 1, "ring of whole stages");
#pragma unroll
    for (int p = 0; p < WG_PF; ++p) load_w(raw[p]);
    load_a(0);
    store_a(0);
    const int nst = (nk + STEPS - 1) / STEPS;
    load_a(min(1, nst - 1));
    lds_barrier();
    // Stages in groups that walk the whole register ring, so its indexes are constants.
    constexpr int GRP = WG_PF / STEPS > 2 ? WG_PF / STEPS : 2;
    for (int s0 = 0; s0 < nst; s0 += GRP) {
#pragma unroll
        for (int g = 0; g < GRP; ++g) {
            const int st = s0 + g;
            if (st >= nst) break;
            // The other slot was last read in stage st - 1, before the barrier.
            if (st + 1 < nst) {
                store_a((g + 1) & 1);
                load_a(min(st + 2, nst - 1));
            }
#pragma unroll
            for (int t = 0; t < STEPS; ++t) {
                const int kk = st * STEPS + t;
                if (kk < nk) step(g & 1, t, kk, raw[(g * STEPS + t) % WG_PF]);
            }
            lds_barrier();
        }
    }

    // Lane l holds D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#pragma unroll
    for (int i = 0; i < WG_TM; ++i)
#pragma unroll
        for (int j = 0; j < WG_TN; ++j) {
            const int n = L.n[j];
            const bool ok = n0 + (WT == WX_Q4 ? 32 * j + lrow : WG_TN * lrow) < a.N;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + 32 * i + 8 * (r >> 2) + 4 * lhi + (r & 3);
                if (m >= a.M || !ok) continue;
                if (a.S > 1) a.part[((int64_t)z * a.M + m) * a.ldp + n] = acc[i][j][r];
                else store_dt(a.Y, (int64_t)m * a.ldy + n, ACT ? wx_activate(acc[i][j][r], a.act) : acc[i][j][r], XT);
            }
        }
}

// Sums the S partial rows in split order and stores Y.
template <int XT>
__global__ void __launch_bounds__(256) wx_reduce_kernel(WxArgs a) {
    const int n = (blockIdx.x * 256 + threadIdx.x) * 4, m = blockIdx.y;
    if (n >= a.N) return;
    const float *p = a.part + (int64_t)m * a.ldp + n;
    float4_t sum = *(const float4_t *)p;
    for (int s = 1; s < a.S; ++s) sum += *(const float4_t *)(p + (int64_t)s * a.M * a.ldp);
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (n + c < a.N) store_dt(a.Y, (int64_t)m * a.ldy + n + c, wx_activate(sum[c], a.act), XT);
}

hipError_t launch_wx_reduce(const WxArgs &a, int x_dt, hipStream_t s) {
    const dim3 grid((a.N + 1023) / 1024, a.M);
    if (x_dt == DT_F16) hipLaunchKernelGGL(wx_reduce_kernel<DT_F16>, grid, dim3(256), 0, s, a);
    else if (x_dt == DT_BF16) hipLaunchKernelGGL(wx_reduce_kernel<DT_BF16>, grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(wx_reduce_kernel<DT_F32>, grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

template <int WT, int XT, bool ACT = false>
static void launch_wx_gemm_t(const WxArgs &a, bool any, dim3 grid, hipStream_t s) {
    if (any) hipLaunchKernelGGL((wx_gemm_kernel<WT, XT, true, ACT>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((wx_gemm_kernel<WT, XT, false, ACT>), grid, dim3(256), 0, s, a);
}
template <int WT>
static void launch_wx_gemm_w(const WxArgs &a, int x_dt, bool any, dim3 grid, hipStream_t s) {
    if (a.act != ACT_NONE && a.S == 1) {          // fused activations: INT4 x fp16 only (wx_supported)
        if constexpr (WT == WX_I4) launch_wx_gemm_t<WT, DT_F16, true>(a, any, grid, s);
    } else if (x_dt == DT_F16) launch_wx_gemm_t<WT, DT_F16>(a, any, grid, s);
    else if (x_dt == DT_BF16) launch_wx_gemm_t<WT, DT_BF16>(a, any, grid, s);
    else launch_wx_gemm_t<WT, DT_F32>(a, any, grid, s);
}

// K splits: one workgroup per CU, at least 8 K steps of 32 each.
int wx_gemm_splits(int64_t M, int64_t K, int64_t N) {
    const int64_t t = ((M + WG_BM - 1) / WG_BM) * ((N + WG_BN - 1) / WG_BN), nks = (K + 31) / 32;
    int S = 1;
    while (t * S * 2 <= 256 && nks / (S * 2) >= 8 && S < 16) S *= 2;
    return S;
}

hipError_t launch_wx_gemm(WxArgs a, int wt, int x_dt, bool any, hipStream_t s) {
    a.tiles_m = (a.M + WG_BM - 1) / WG_BM;
    a.tiles_n = (a.N + WG_BN - 1) / WG_BN;
    const dim3 grid((unsigned)(a.tiles_m * a.tiles_n), 1, a.S);
    if (wt == WX_Q4) launch_wx_gemm_w<WX_Q4>(a, x_dt, any, grid, s);
    else if (wt == WX_I4) launch_wx_gemm_w<WX_I4>(a, x_dt, any, grid, s);
    else launch_wx_gemm_w<WX_I8>(a, x_dt, any, grid, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.S == 1) return e;
    return launch_wx_reduce(a, x_dt, s);
}

}  // namespace mcq4
