// Any-activation prefill matmul (wx_common.h): 128 x 256 tiles, one 8-wave
// workgroup per CU.  Waves (c, ph): four column groups of 64 x two K phases, each
// wave a 128 x 64 tile (MFMA 32x32, 128 fp32 accumulators) over its phase's half
// of every stage; two waves per SIMD, so one's dequant and waits run under the
// other's MFMAs.  The two phases are summed in LDS at the end.
//
//   * Weights go from global memory straight into registers, up to three K steps of
//     32 ahead: each weight is read and dequantized once per workgroup, and no
//     alignment beyond the format's own is needed (any N, any row offset).  A
//     ring slot is loaded one step after its last use and no branch stands
//     between loads and MFMAs: otherwise the compiler moves values still in
//     flight between registers, waiting for them.
//   * Activations: one stage (256 bytes of each of the 128 rows: four K steps in 16
//     bits, two in fp32) goes through registers into one of two LDS slots, loaded
//     a whole stage ahead; chunk c of row r sits at c ^ (r & 7), so the 16-byte
//     operand reads are free of bank conflicts.  ANY: activations that are not
//     16-byte aligned, or a K that is no multiple of 32, are read element by
//     element, zero past K.
//   * 16-bit activations: v_mfma_f32_32x32x16_{f16,bf16}, a B operand feeding
//     four MFMAs.  fp32: v_mfma_f32_32x32x2_f32, weights kept in fp32, 64 x 256 tiles: the
//     other half of the accumulators holds the running sums, to which each step's 32
//     products are added as a sum of their own (error against 64 bits, K = 4096: 1.3e-7 of
//     the result; 5e-7 in one chain of K / 2, 3.9e-7 in eight of K / 8).
//   * Split K (grid.z) for outputs with few tiles: fp32 partial rows summed in
//     split order by wx_reduce_kernel.
//
// Measured: INT4 x bf16 M = 256 4096x11008 60.9 us (one thread per column: 8165), INT4 x
// fp32 243.2, q4_0 x fp16 M = 300 11008x4101 83.9.  INT4 in 16 bits is bound by waits
// (counters: MFMA busy 15 %, 44 % of the wave cycles waiting, LDS conflicts 28 % of the
// LDS cycles); fp32 by the fp32 MFMA, whose library rate is 153 TFLOP/s here (95 at M =
// 256, 108 at 512x4096x4096).  Operands prepared one step ahead of their MFMAs: 61.5 us.
#include <algorithm>
#include <type_traits>

#include "wx_common.h"

namespace mcq4 {

constexpr int WG_BN = 256, WG_TN = 2;
constexpr int wg_tm(int xt) { return xt == DT_F32 ? 2 : 4; }   // row tiles of 32
constexpr int WG_SLOT = 128 * 256;               // 128 rows (fp32: 64)
constexpr size_t WG_LDS = 4 * 2 * 2 * WG_TN * 16 * 64 * 4;   // phase sum: 4 column groups x 2 halves, 128 KB (the loop: 64 + scratch)
static_assert(WG_LDS >= 2 * WG_SLOT + 8 * wx_scratch(WX_I8) && WG_LDS <= 160 * 1024, "LDS budget");

template <int WT, int XT, bool SZ32, bool ANY, bool ACT>
__global__ void __launch_bounds__(512, 2) wx_gemm_kernel(WxArgs a) {
    constexpr int ES = XT == DT_F32 ? 4 : 2;
    constexpr int SPW = XT == DT_F32 ? 1 : 2;    // K steps of 32 per wave and stage
    constexpr int TM = wg_tm(XT), BM = 32 * TM;
    constexpr int R = 4;                         // ring slots: R - 1 steps in flight
    extern __shared__ __attribute__((aligned(16))) uint8_t sA[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wc = wave & 3, ph = wave >> 2;
    const int lrow = lane & 31, lhi = lane >> 5;

    const int bid = blockIdx.x, gx = gridDim.x;
    int tile_id = bid;
    if (gx % 8 == 0) tile_id = (bid % 8) * (gx / 8) + bid / 8;   // consecutive tiles on one XCD
    const int m0 = (tile_id % a.tiles_m) * BM, n0 = (tile_id / a.tiles_m) * WG_BN + 64 * wc;
    const int nks = (a.K + 31) / 32;
    const int z = blockIdx.z;
    const int k_lo = (int)((int64_t)nks * z / a.S), nk = (int)((int64_t)nks * (z + 1) / a.S) - k_lo;
    const int nst = (nk + 2 * SPW - 1) / (2 * SPW);

    const WxLane<WT, WG_TN> L = wx_lane<WT, WG_TN>(a, n0, lane);

    // Activation copies: thread t moves chunks (row t / 16 + 32 u, chunk t % 16), u < TM.
    const uint8_t *xrow[TM];
    const int xc = tid & 15;
#pragma unroll
    for (int u = 0; u < TM; ++u)
        xrow[u] = (const uint8_t *)a.X + (int64_t)min(m0 + (tid >> 4) + 32 * u, a.M - 1) * a.ldx * ES;
    uint4_t xs[TM];
    auto load_a = [&](int st) {
        const int k = (k_lo + min(st, nst - 1) * (2 * SPW)) * 32 + xc * (16 / ES);
#pragma unroll
        for (int u = 0; u < TM; ++u) {
            if constexpr (ANY) xs[u] = wx_load_x_any<XT>(xrow[u], k, a.K);
            // Past the split's end (a last stage that is not whole): any valid chunk, no MFMA uses it.
            else xs[u] = *(const uint4_t *)(xrow[u] + (int64_t)min(k, a.K - 16 / ES) * ES);
        }
    };
    auto store_a = [&](int slot) {
#pragma unroll
        for (int u = 0; u < TM; ++u) {
            const int r = (tid >> 4) + 32 * u;
            *(uint4_t *)(sA + slot * WG_SLOT + r * 256 + ((xc ^ (r & 7)) << 4)) = XT == DT_F32 ? xs[u] : wx_order<WT>(xs[u]);
        }
    };
    auto read_a = [&](int slot, int i, int chunk) {
        return *(const uint4_t *)(sA + slot * WG_SLOT + (32 * i + lrow) * 256 + ((chunk ^ (lrow & 7)) << 4));
    };

    // This wave's u-th K step (of the split's nk) and its weights.
    auto kstep = [&](int u) { return u / SPW * (2 * SPW) + ph * SPW + u % SPW; };
    WxFly<WT, WG_TN> raw[R];
    uint8_t *const scratch = sA + 2 * WG_SLOT + wave * wx_scratch(WT);
    auto load_w = [&](WxFly<WT, WG_TN> &r, int u) {
        wx_load<WT, WG_TN, SZ32, ANY && WT != WX_Q4>(r, a, L, k_lo + min(kstep(u), nk - 1), lane);
    };

    std::conditional_t<XT == DT_F32, float[TM][WG_TN][16], float16_t[TM][WG_TN]> acc;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < WG_TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    auto step = [&](int slot, int t, int u, const WxFly<WT, WG_TN> &f) {
        const WxRaw<WT, WG_TN> r = wx_ready<WT, WG_TN, false>(f, scratch, lane);
        const int valid = a.K - (k_lo + kstep(u)) * 32 - 16 * lhi;
        const uint16_t *d = nullptr;
        if constexpr (WT == WX_Q4) d = r.d;
        if constexpr (XT == DT_F32) {
            // A step's 32 products are summed from zero and then added: chains of 32 and K / 64.
            float w[WG_TN][16];
            float16_t part[TM][WG_TN];
            wx_if_finite<WT, XT, WG_TN>(d, [&](auto fin) {
#pragma unroll
                for (int j = 0; j < WG_TN; ++j)
                    wx_values<WT, XT, WG_TN, SZ32, ANY, decltype(fin)::value>(r, j, a.sz_dt, valid, w[j]);
            });
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float4_t x[TM][2];
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int q = 0; q < 2; ++q) x[i][q] = bitcast<float4_t>(read_a(slot, i, 8 * ph + 4 * lhi + 2 * h + q));
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    const int e = wx_slot<WT>(s);
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < WG_TN; ++j)
                            part[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i][e / 4][e % 4], w[j][8 * h + s],
                                                                              h + s ? part[i][j] : float16_t{}, 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < WG_TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        float v = acc[i][j][r] + part[i][j][r];
                        asm volatile("" : "+v"(v));   // else the add sinks to the next step, part with it
                        acc[i][j][r] = v;
                    }
        } else {
            uint4_t B[WG_TN][2];
            wx_if_finite<WT, XT, WG_TN>(d, [&](auto fin) {
#pragma unroll
                for (int j = 0; j < WG_TN; ++j)
                    wx_operands<WT, XT, WG_TN, SZ32, ANY, decltype(fin)::value>(r, j, a.sz_dt, valid, B[j]);
            });
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    const uint4_t x = read_a(slot, i, 8 * ph + 4 * t + 2 * lhi + ks);
#pragma unroll
                    for (int j = 0; j < WG_TN; ++j) acc[i][j] = wx_mfma<XT>(x, B[j][ks], acc[i][j]);
                }
        }
    };

#pragma unroll
    for (int p = 0; p < R - 1; ++p) load_w(raw[p], p);
    load_a(0);
    store_a(0);
    load_a(1);
    lds_barrier();
    // Stages in groups of four steps, so the ring's indexes are constants; `guard`: the
    // last group, whose stages and steps may lie past the end.
    constexpr int GRP = 4 / SPW;
    auto group = [&](auto guard, int s0) {
#pragma unroll
        for (int g = 0; g < GRP; ++g) {
            const int st = s0 + g;
            if (decltype(guard)::value && st >= nst) break;
            // The other slot was last read in stage st - 1, before the barrier.
            store_a((g + 1) & 1);
            load_a(st + 2);
#pragma unroll
            for (int t = 0; t < SPW; ++t) {
                const int p = g * SPW + t, u = st * SPW + t;
                load_w(raw[(p + R - 1) % R], u + R - 1);
                __builtin_amdgcn_sched_barrier(0);
                if (!decltype(guard)::value || kstep(u) < nk) step(g & 1, t, u, raw[p % R]);
            }
            lds_barrier();
        }
    };
    int s0 = 0;
    for (; (s0 + GRP) * 2 * SPW <= nk; s0 += GRP) group(std::false_type{}, s0);
    if (s0 < nst) group(std::true_type{}, s0);

    // Phase sum: each wave gives the other phase's half of its rows
    // away and adds the other's share of its own.
    constexpr int H = TM / 2;
    static_assert(GRP % 2 == 0 && TM % 2 == 0, "slot parity; halves of the row tiles");
    float *const sum = (float *)sA + (wc * 2 + ph) * (H * WG_TN * 16 * 64) + lane;
    float *const mine = (float *)sA + (wc * 2 + (1 - ph)) * (H * WG_TN * 16 * 64) + lane;
#pragma unroll
    for (int i = 0; i < H; ++i)
#pragma unroll
        for (int j = 0; j < WG_TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[((i * WG_TN + j) * 16 + r) * 64] = ph ? acc[i][j][r] : acc[H + i][j][r];
    lds_barrier();
    // Lane l holds D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#pragma unroll
    for (int i = 0; i < H; ++i)
#pragma unroll
        for (int j = 0; j < WG_TN; ++j) {
            const int n = L.n[j];
            const bool ok = n0 + (WT == WX_Q4 ? 32 * j + lrow : 16 * (lrow >> 3)) < a.N;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + 32 * H * ph + 32 * i + 8 * (r >> 2) + 4 * lhi + (r & 3);
                const float o = mine[((i * WG_TN + j) * 16 + r) * 64];
                const float v = ph ? o + acc[H + i][j][r] : acc[i][j][r] + o;   // phase 0 + phase 1
                if (m >= a.M || !ok) continue;
                if (a.S > 1) a.part[((int64_t)z * a.M + m) * a.ldp + n] = v;
                else store_dt(a.Y, (int64_t)m * a.ldy + n, ACT ? wx_activate(v, a.act) : v, XT);
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

template <int WT, int XT, bool SZ32, bool ANY, bool ACT>
static hipError_t launch_wx_gemm_k(const WxArgs &a, dim3 grid, hipStream_t s) {
    if (hipError_t e = hipFuncSetAttribute((const void *)wx_gemm_kernel<WT, XT, SZ32, ANY, ACT>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)WG_LDS))
        return e;
    hipLaunchKernelGGL((wx_gemm_kernel<WT, XT, SZ32, ANY, ACT>), grid, dim3(512), WG_LDS, s, a);
    return hipGetLastError();
}
template <int WT, int XT, bool SZ32, bool ACT = false>
static hipError_t launch_wx_gemm_t(const WxArgs &a, bool any, dim3 grid, hipStream_t s) {
    return any ? launch_wx_gemm_k<WT, XT, SZ32, true, ACT>(a, grid, s) : launch_wx_gemm_k<WT, XT, SZ32, false, ACT>(a, grid, s);
}
template <int WT, bool SZ32>
static hipError_t launch_wx_gemm_s(const WxArgs &a, int x_dt, bool any, dim3 grid, hipStream_t s) {
    // Fused activations: INT4 x fp16 only (wx_supported); with a K split the reduction applies them.
    if constexpr (WT == WX_I4)
        if (a.act != ACT_NONE && a.S == 1) return launch_wx_gemm_t<WT, DT_F16, SZ32, true>(a, any, grid, s);
    if (x_dt == DT_F16) return launch_wx_gemm_t<WT, DT_F16, SZ32>(a, any, grid, s);
    if (x_dt == DT_BF16) return launch_wx_gemm_t<WT, DT_BF16, SZ32>(a, any, grid, s);
    return launch_wx_gemm_t<WT, DT_F32, SZ32>(a, any, grid, s);
}

// K splits, at least 8 K steps of 32 each.  16 bits: as many as keep one workgroup per
// CU.  fp32 is bound by its MFMAs, so a last round of workgroups that leaves CUs idle
// costs in full: the split with the least rounds(t S) / S, plus the partials' traffic (8
// bytes an output and split at about 5 TB/s against 2 K operations at about 100 TFLOP/s:
// 80 / K of a full round).  us, at most one per CU / this: 256x4096x11008 (172 tiles)
// 279.6 / 237.0, 512x4096x4100 (136 tiles) 289.4 / 202.6.
int wx_gemm_splits(int x_dt, int64_t M, int64_t K, int64_t N) {
    const int64_t bm = 32 * wg_tm(x_dt), t = ((M + bm - 1) / bm) * ((N + WG_BN - 1) / WG_BN), nks = (K + 31) / 32;
    if (x_dt != DT_F32 || t >= 1024) return (int)std::max<int64_t>(1, std::min<int64_t>({256 / t, nks / 8, 16}));
    int best = 1;
    double least = 0;
    for (int S = 1; S <= 16 && (S == 1 || nks / S >= 8); ++S) {
        const double cost = (double)((t * S + 255) / 256) / S + S * (t / 256.0) * (80.0 / (double)K);
        if (S == 1 || cost < least) {
            best = S;
            least = cost;
        }
    }
    return best;
}

hipError_t launch_wx_gemm(WxArgs a, int wt, int x_dt, bool any, hipStream_t s) {
    const int bm = 32 * wg_tm(x_dt);
    a.tiles_m = (a.M + bm - 1) / bm;
    a.tiles_n = (a.N + WG_BN - 1) / WG_BN;
    const dim3 grid((unsigned)(a.tiles_m * a.tiles_n), 1, a.S);
    const bool sz32 = a.sz_dt == DT_F32;
    const hipError_t e = wt == WX_Q4   ? launch_wx_gemm_s<WX_Q4, false>(a, x_dt, any, grid, s)
                         : wt == WX_I4 ? (sz32 ? launch_wx_gemm_s<WX_I4, true>(a, x_dt, any, grid, s)
                                               : launch_wx_gemm_s<WX_I4, false>(a, x_dt, any, grid, s))
                                       : (sz32 ? launch_wx_gemm_s<WX_I8, true>(a, x_dt, any, grid, s)
                                               : launch_wx_gemm_s<WX_I8, false>(a, x_dt, any, grid, s));
    if (e != hipSuccess || a.S == 1) return e;
    return launch_wx_reduce(a, x_dt, s);
}

}  // namespace mcq4
