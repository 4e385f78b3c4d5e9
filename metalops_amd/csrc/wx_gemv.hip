// q4_0 decode for any activation dtype, M <= 16 (wx_common.h): one workgroup owns
// 16 TN neighbouring columns, its waves split K and sum through LDS in wave order.
//
//   * MFMA 16x16 with a K step of four blocks: lane (c = l % 16, g = l / 16) loads
//     block kb + g of column c whole (18 contiguous bytes, unaligned register
//     loads) and the same 32 activations of row min(c, M - 1); MFMA i takes
//     elements 8 i .. +7 of each lane's block, so the K order is a permutation
//     of the real one, the same for both operands.
//   * Each weight is rounded once to X's dtype (the dtype's own semantics), which
//     is what bounds the kernel beside the weight bytes: about two VALU instructions
//     per weight for bf16.  So the columns are spread over the CUs
//     as evenly as 16-column groups allow (TN below), with no K split over
//     workgroups and one launch.
//   * fp32: v_mfma_f32_16x16x4_f32, half the matrix time of the 32-row form;
//     64 products at a time are summed from zero, then added (error as in wx_gemm).
//
// Measured: fp16 M = 1 / 16 4096x12289 12.4 / 15.7 us (q4_skinny 16.7 / 19.8), fp32 M = 8
// 4096x11008 22.7.  Fewer VALU per weight (3.3 to 2.1) changed nothing: the unaligned
// 16-byte loads at 18-byte stride take the time.
#include "wx_common.h"

namespace mcq4 {

template <int XT, int TN, int NW, bool ANY>
__global__ void __launch_bounds__(NW * 64) wx_gemv_kernel(WxArgs a) {
    constexpr int ES = XT == DT_F32 ? 4 : 2;
    constexpr int XV = 32 * ES / 16;             // 16-byte activation loads per block
    __shared__ float red[NW][TN][4][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (16 * TN);
    const int nb = a.K / QK, nst = (nb + 3) / 4;
    const int s_lo = (int)((int64_t)nst * wave / NW), ns = (int)((int64_t)nst * (wave + 1) / NW) - s_lo;

    uint32_t off[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) off[j] = (uint32_t)(min(n0 + 16 * j + c, a.N - 1) - min(n0, a.N - 1)) * BLOCK_BYTES;
    const uint8_t *const xrow = (const uint8_t *)a.X + (int64_t)min(c, a.M - 1) * a.ldx * ES;

    struct Step {
        uint4_t q[TN], x[XV];
        uint16_t d[TN];
    } ring[2];
    auto load = [&](Step &p, int u) {
        // Blocks past K: the last one again (step() drops it).
        const int kb = min(4 * (s_lo + min(u, ns - 1)) + g, nb - 1);
        const uint8_t *base = a.W + ((int64_t)kb * a.N + min(n0, a.N - 1)) * BLOCK_BYTES;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            p.d[j] = load_u<uint16_t>(base + off[j]);
            p.q[j] = load_u<uint4_t>(base + off[j] + 2);
        }
#pragma unroll
        for (int v = 0; v < XV; ++v) {
            const int k = kb * QK + v * (16 / ES);
            if constexpr (ANY) p.x[v] = wx_load_x_any<XT>(xrow, k, a.K);
            else p.x[v] = *(const uint4_t *)(xrow + (int64_t)k * ES);
        }
    };

    float4_t acc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[j] = float4_t{0.f, 0.f, 0.f, 0.f};

    auto step = [&](Step &p, int u) {
        if (4 * (s_lo + u) + 3 >= nb) {          // K % 128 != 0: drop the blocks past K
            const bool ok = 4 * (s_lo + u) + g < nb;
#pragma unroll
            for (int v = 0; v < XV; ++v)
#pragma unroll
                for (int e = 0; e < 4; ++e) p.x[v][e] = ok ? p.x[v][e] : 0u;
#pragma unroll
            for (int j = 0; j < TN; ++j) p.d[j] = ok ? p.d[j] : (uint16_t)0;
        }
        if constexpr (XT != DT_F32) {
#pragma unroll
            for (int v = 0; v < XV; ++v) p.x[v] = wx_order<WX_Q4>(p.x[v]);
        }
        wx_if_finite<WX_Q4, XT, TN>(p.d, [&](auto fin) {
            constexpr bool FIN = decltype(fin)::value;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                WxRaw<WX_Q4, 1> r;
                r.d[0] = p.d[j];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    r.q[0][0] = p.q[j][2 * h]; r.q[0][1] = p.q[j][2 * h + 1];
                    if constexpr (XT == DT_F32) {
                        float w[16];
                        float4_t part;       // 64 products, summed from zero
                        wx_values<WX_Q4, XT, 1, false, false, FIN>(r, 0, 0, 16, w);
#pragma unroll
                        for (int s = 0; s < 16; ++s) {
                            const int e = wx_slot<WX_Q4>(s);
                            part = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(p.x[4 * h + e / 4][e % 4]), w[s],
                                                                        s ? part : float4_t{}, 0, 0, 0);
                        }
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            float v = acc[j][r] + part[r];
                            asm volatile("" : "+v"(v));
                            acc[j][r] = v;
                        }
                    } else {
                        uint4_t B[2];
                        wx_operands<WX_Q4, XT, 1, false, false, FIN>(r, 0, 0, 16, B);
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks) acc[j] = wx_mfma16<XT>(p.x[2 * h + ks], B[ks], acc[j]);
                    }
                }
            }
        });
    };

    if (ns > 0) {
        load(ring[0], 0);
        for (int u0 = 0; u0 < ns; u0 += 2) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                if (u0 + p >= ns) break;
                load(ring[1 - p], u0 + p + 1);   // into the slot step u0 + p - 1 has left
                __builtin_amdgcn_sched_barrier(0);
                step(ring[p], u0 + p);
            }
        }
    }

    // Lane l holds rows 4 (l / 16) + i of column l % 16.
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][j][i][lane] = acc[j][i];
    __syncthreads();
    for (int v = tid; v < TN * 256; v += NW * 64) {
        const int j = v >> 8, i = (v >> 6) & 3, m = 4 * ((v >> 4) & 3) + i, n = n0 + 16 * j + (v & 15);
        if (m >= a.M || n >= a.N) continue;
        float sum = red[0][j][i][v & 63];
#pragma unroll
        for (int w = 1; w < NW; ++w) sum += red[w][j][i][v & 63];
        store_dt(a.Y, (int64_t)m * a.ldy + n, sum, XT);
    }
}

template <int XT, int TN>
static hipError_t launch_wx_gemv_t(const WxArgs &a, bool any, hipStream_t s) {
    // fp32 steps, and bf16 ones of 64 columns, need more than the 128 registers a 16-wave workgroup has.
    constexpr int NW = XT == DT_F32 || (XT == DT_BF16 && TN == 4) ? 8 : 16;
    const dim3 grid((a.N + 16 * TN - 1) / (16 * TN));
    if (any) hipLaunchKernelGGL((wx_gemv_kernel<XT, TN, NW, true>), grid, dim3(NW * 64), 0, s, a);
    else hipLaunchKernelGGL((wx_gemv_kernel<XT, TN, NW, false>), grid, dim3(NW * 64), 0, s, a);
    return hipGetLastError();
}

template <int XT>
static hipError_t launch_wx_gemv_x(const WxArgs &a, int tn, bool any, hipStream_t s) {
    switch (tn) {
        case 1: return launch_wx_gemv_t<XT, 1>(a, any, s);
        case 2: return launch_wx_gemv_t<XT, 2>(a, any, s);
        case 3: return launch_wx_gemv_t<XT, 3>(a, any, s);
        default: return launch_wx_gemv_t<XT, 4>(a, any, s);
    }
}

// Column groups per workgroup: the fewest 16-column groups on the busiest of 256
// CUs (one workgroup each at a time), the wider workgroup among equals.
static int wx_gemv_tn(int64_t N) {
    const int64_t t = (N + 15) / 16;
    int best = 1;
    int64_t cost = INT64_MAX;
    for (int tn = 1; tn <= 4; ++tn) {
        const int64_t rounds = ((t + tn - 1) / tn + 255) / 256;
        if (rounds * tn <= cost) { cost = rounds * tn; best = tn; }
    }
    return best;
}

hipError_t launch_wx_gemv(const WxArgs &a, int x_dt, bool any, hipStream_t s) {
    const int tn = wx_gemv_tn(a.N);
    if (x_dt == DT_F16) return launch_wx_gemv_x<DT_F16>(a, tn, any, s);
    if (x_dt == DT_BF16) return launch_wx_gemv_x<DT_BF16>(a, tn, any, s);
    return launch_wx_gemv_x<DT_F32>(a, tn, any, s);
}

}  // namespace mcq4
