// q4_0 for 17..64 rows of 16-bit activations, aligned weights (N % 8 == 0): one
// 8-wave workgroup owns 64 columns and 16 RT rows, its waves split K and sum through
// LDS in wave order.
//
//   * Between the decode kernels (16 rows a block, activations in registers) and the
//     128-row prefill tiles, whose fixed part and idle rows cost more than the
//     weights' bytes here.  Each weight is read and dequantized once.
//   * Weights: each wave copies the 1152 bytes of its 64 columns' K block into a
//     private LDS ring, up to three steps ahead (the register loads of wx_skinny, 8 bytes
//     per lane at 18-byte stride, take several times the copies' time).
//   * Activations: copied beside the weights into the ring, 16 rows x 64 bytes per
//     copy, four neighbouring lanes on one row.  (Loaded straight into the operand
//     registers, where neighbouring lanes hold different rows, each lane is a
//     cache request of its own: 48 rows of 4096x14336 took 20.4 us, 14.3 with every
//     lane on row 0.)  Chunk c of row r sits at c ^ ((r / 2) & 3), so the operand
//     reads are free of bank conflicts.  Rows past M repeat the last one.
//   * Split K over workgroups (blockIdx.y) where the columns alone leave CUs idle:
//     splits of a tile share an XCD, split 0 sums their partials from its L2 once
//     their flags show them stored, as in q4_gemv_span.hip (above 32 rows, or with
//     MCQ4_XCD_LOCAL=0, wx_reduce_kernel sums).
//   * fp16 up to 32 rows: the decode kernels' arithmetic, sum x (q - 8) of a block
//     exact in the MFMA and scaled by d in fp32.  Otherwise the weight (q - 8) d is
//     rounded to the activations' dtype first, as the prefill kernels do.
//   * MFMA lane rows g = 0..3 take K quarters 0, 2, 1, 3 of a block (both operands):
//     fewer LDS bank conflicts on the nibble reads.
//
// Measured (graph replays, fp16): 4096x14336 M = 17 / 32 / 48 / 64 12.3 / 13.1 / 16.7 /
// 18.2 us, against 17.0 / 19.2 (q4_gemvm, two row blocks) and 27.6 / 27.5 (q4_gemm6);
// 14336x4096 M = 24 / 64 14.6 / 21.2 against 20.0 / 31.0; 4096x4096 M = 24 8.6
// against 9.3.  A plain read of the weights' pattern takes about 6.5.
#include <atomic>

#include "wx_common.h"

namespace mcq4 {

MCQ4_SPLIT_FALLBACK_COUNTER(wx_mid_split_fallbacks)

constexpr int WM_NW = 8, WM_CT = 4;            // waves; 16-column tiles
constexpr int WM_SMAX = 8;                     // K splits at most
// K steps in flight beside the one in work (LDS: one workgroup per CU).
constexpr int wm_depth(int rt) { return rt == 4 ? 2 : 3; }
constexpr int WM_RAW = 1280;                   // 1152 + the remainder copy's idle lanes and the read overhang
constexpr int wm_slot(int rt) { return 1024 * rt + WM_RAW; }
constexpr size_t wm_lds(int rt) {
    const size_t ring = (size_t)WM_NW * (wm_depth(rt) + 1) * wm_slot(rt), sum = (size_t)WM_NW * rt * WM_CT * 256 * 4;
    return (ring > sum ? ring : sum) + 16;     // + the split mask
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t wm_rsrc(const void *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, bytes, 0x00020000);
}
__device__ __forceinline__ void wm_copy(__amdgpu_buffer_rsrc_t rs, uint8_t *dst, uint32_t so, uint32_t vo16, uint32_t vo4) {
    // (The instruction's immediate offset would move the LDS destination too.)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)dst, 16, vo16, so, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)(dst + 1024), 4, vo4, so, 0, 0);
}
__device__ __forceinline__ void wm_copy_x(__amdgpu_buffer_rsrc_t rs, uint8_t *dst, uint32_t so, uint32_t vo) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)dst, 16, vo, so, 0, 0);
}

template <int XT, int RT>
__global__ void __launch_bounds__(WM_NW * 64) wx_mid_kernel(WxArgs a) {
    constexpr int D = wm_depth(RT), SLOT = wm_slot(RT);
    constexpr int PER = 2 + RT;                  // vector-memory instructions per step
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4, kq = ((g & 1) << 1) | (g >> 1);
    const int z = blockIdx.y;
    int tile = blockIdx.x;
    uint32_t fb = 0;                             // the tile's split flags as the launch starts
    if (a.flags) {
        // XCD-renumbered, grid.x a multiple of 8: every split of a tile on one XCD.
        tile = (tile & 7) * ((int)gridDim.x >> 3) + (tile >> 3);
        if (tile * 64 >= a.N) return;            // grid padding
        if (wave == 0 && lane < a.S)
            fb = __hip_atomic_load(a.flags + tile * a.S + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int n0 = tile * 64;
    const int nks = a.K / QK;
    const int ws = z * WM_NW + wave, wt = a.S * WM_NW;
    const int k_lo = (int)((int64_t)nks * ws / wt), nk = (int)((int64_t)nks * (ws + 1) / wt) - k_lo;
    uint8_t *const ring = smem + wave * ((D + 1) * SLOT);

    // Columns past N: the lane re-reads the row's last bytes, whose outputs are not stored.
    const uint32_t valid = (uint32_t)min(64, a.N - n0) * BLOCK_BYTES;
    const uint32_t vo16 = min(16u * lane, valid - 16), vo4 = min(1024u + 4u * min(lane, 31), valid - 4);
    const uint32_t row_bytes = (uint32_t)a.N * BLOCK_BYTES;
    const __amdgpu_buffer_rsrc_t w_rs = wm_rsrc(a.W, 0x7fffffff), x_rs = wm_rsrc(a.X, 0x7fffffff);
    // Lane l copies chunk (l % 4) ^ ((l / 8) & 3) of row 16 i + l / 4.
    uint32_t xo[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
        xo[i] = (uint32_t)(min(16 * i + (lane >> 2), a.M - 1) * a.ldx + 8 * ((lane & 3) ^ ((lane >> 3) & 3))) * 2;

    auto issue = [&](int slot, int kk) {
        const uint32_t kb = (uint32_t)(k_lo + min(kk, nk - 1));
        uint8_t *const dst = ring + slot * SLOT;
#pragma unroll
        for (int i = 0; i < RT; ++i) wm_copy_x(x_rs, dst + 1024 * i, kb * (QK * 2), xo[i]);
        wm_copy(w_rs, dst + 1024 * RT, kb * row_bytes + (uint32_t)n0 * BLOCK_BYTES, vo16, vo4);
        __builtin_amdgcn_sched_barrier(0);
    };

    float4_t acc[RT][WM_CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < WM_CT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

    const int qoff = 18 * c + 2 + 4 * kq;
    const uint32_t qal = (uint32_t)(qoff & ~3), qsh = (uint32_t)(qoff & 3) * 8;
    const int xoff = 64 * c + 16 * (kq ^ ((c >> 1) & 3));
    auto step = [&](int slot) {
        const lds_u8 *Xs = lds_ptr(lds_addr(ring + slot * SLOT)), *Rs = Xs + 1024 * RT;
        uint32_t q[WM_CT];
        uint16_t d[WM_CT];
#pragma unroll
        for (int j = 0; j < WM_CT; ++j) {
            const lds_u32 *qp = (const lds_u32 *)(Rs + qal + j * (16 * 18));
            q[j] = __builtin_amdgcn_alignbit(qp[1], qp[0], qsh);
            d[j] = *(const lds_u16 *)(Rs + 18 * c + j * (16 * 18));
        }
        uint4_t x[RT];
#pragma unroll
        for (int i = 0; i < RT; ++i) x[i] = wx_order<WX_Q4>(bitcast<uint4_t>(*(const lds_half8 *)(Xs + xoff + 1024 * i)));
        if constexpr (XT == DT_F16 && RT == 2) {
#pragma unroll
            for (int j = 0; j < WM_CT; ++j) {
                const float df = (float)bitcast<_Float16>(d[j]);
                const uint4_t B = q4_exact8(q[j]);
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const float4_t t = wx_mfma16<XT>(x[i], B, float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(df, t[r], acc[i][j][r]);
                }
            }
            return;
        }
        wx_if_finite<WX_Q4, XT, WM_CT>(d, [&](auto fin) {
#pragma unroll
            for (int j = 0; j < WM_CT; ++j) {
                const uint4_t B = q4_operand8<XT, decltype(fin)::value>(q[j], d[j]);
#pragma unroll
                for (int i = 0; i < RT; ++i) acc[i][j] = wx_mfma16<XT>(x[i], B, acc[i][j]);
            }
        });
    };

    if (nk > 0) {
#pragma unroll
        for (int p = 0; p < D; ++p) issue(p, p);
        for (int k0 = 0; k0 < nk; k0 += D + 1) {
#pragma unroll
            for (int p = 0; p <= D; ++p) {
                if (k0 + p >= nk) break;
                issue((p + D) % (D + 1), k0 + p + D);   // the slot step k - 1 has left
                wait_vmcnt<D * PER>();
                step(p);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
        }
        wait_vmcnt<0>();                         // the ring's last copies, before the sums reuse it
    }
    __syncthreads();

    // Wave sums: lane l holds rows 4 (l / 16) + r, column l % 16 of each 16 x 16 tile.
    constexpr int T = RT * WM_CT;
    float *const red = (float *)smem;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < WM_CT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[((wave * T + i * WM_CT + j) * 4 + r) * 64 + lane] = acc[i][j][r];
    __syncthreads();
    // Thread: column l of the 64, rows 8 u + wave.
    auto own = [&](int u) {
        const int v = tid + u * (WM_NW * 64), mr = v >> 6, i = mr >> 4, j = (v >> 4) & 3, gg = (mr >> 2) & 3, r = mr & 3;
        const float *p = red + ((i * WM_CT + j) * 4 + r) * 64 + 16 * gg + (v & 15);
        float sum = p[0];
#pragma unroll
        for (int w = 1; w < WM_NW; ++w) sum += p[w * T * 256];
        return sum;
    };
    constexpr int U = T * 256 / (WM_NW * 64);    // outputs per thread
    const int n = n0 + lane;
    if (z != 0 || !a.flags) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int mr = 8 * u + wave;
            if (mr >= a.M || n >= a.N) continue;
            const float sum = own(u);
            if (a.S > 1) a.part[((int64_t)z * a.M + mr) * a.ldp + n] = sum;
            else store_dt(a.Y, (int64_t)mr * a.ldy + n, sum, XT);
        }
        if (!a.flags) return;
        // A flag is one word per (tile, split) written only by that split, which adds 8 to
        // the value it held when the launch started and puts its XCD id in the low 3
        // bits: whatever other kernels left there between launches, during one it
        // holds its starting value or this launch's.
        wait_vmcnt<0>();
        __syncthreads();
        if (wave == 0 && lane == z)
            __hip_atomic_store(a.flags + tile * a.S + z, (fb & ~7u) + 8u + xcc_id(), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        return;
    }
    // Split 0: wait (at most a.spin polls) for the other splits' flags, then add their
    // partials in split order from the XCD's L2; a split whose flag comes from another
    // XCD, or not in time, is recomputed from the inputs.
    uint32_t *const mask = (uint32_t *)(smem + wm_lds(RT) - 16);
    if (wave == 0) {
        const uint32_t xcc = xcc_id();
        const bool mine = lane >= 1 && lane < a.S;
        const uint32_t want = (fb & ~7u) + 8u;
        uint32_t v = 0;
        bool seen = !mine;
        for (uint32_t it = 0; it < a.spin; ++it) {
            if (!seen) {
                v = __hip_atomic_load(a.flags + tile * a.S + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                seen = (v & ~7u) == want;
            }
            if (__all(seen)) break;
            __builtin_amdgcn_s_sleep(1);
        }
        const uint64_t good = __ballot(mine && seen && (v & 7u) == xcc);
        if (lane == 0) {
            *mask = ((uint32_t)good | 1u) & ~(a.foreign & ~1u);
            if (*mask != (1u << a.S) - 1) note_split_fallback();
        }
    }
    __syncthreads();
    const uint32_t local = *mask;
    float pv[U][WM_SMAX - 1];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 1; q < WM_SMAX; ++q) {
            const int mr = min(8 * u + wave, a.M - 1);
            if (q < a.S && ((local >> q) & 1))
                pv[u][q - 1] = load_l2_f32(a.part, (int)((((int64_t)q * a.M + mr) * a.ldp + min(n, a.N - 1)) * 4));
        }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int mr = 8 * u + wave;
        if (mr >= a.M || n >= a.N) continue;
        float sum = own(u);
#pragma unroll
        for (int q = 1; q < WM_SMAX; ++q) {
            if (q >= a.S) break;
            float v = pv[u][q - 1];
            if (!((local >> q) & 1))
                v = q4_dot_range<XT == DT_BF16>((const _Float16 *)a.X + (int64_t)mr * a.ldx, a.W, a.N, n,
                                                (int)((int64_t)nks * q / a.S), (int)((int64_t)nks * (q + 1) / a.S));
            sum += v;
        }
        store_dt(a.Y, (int64_t)mr * a.ldy + n, sum, XT);
    }
}

template <int XT, int RT>
static hipError_t launch_wx_mid_t(const WxArgs &a, hipStream_t s) {
    constexpr size_t lds = wm_lds(RT);
    static std::atomic<uint64_t> done{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(done.load(std::memory_order_acquire) & bit)) {
        e = hipFuncSetAttribute((const void *)wx_mid_kernel<XT, RT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        done.fetch_or(bit, std::memory_order_acq_rel);
    }
    const int tiles = (a.N + 63) / 64, gx = a.flags ? (tiles + 7) / 8 * 8 : tiles;
    hipLaunchKernelGGL((wx_mid_kernel<XT, RT>), dim3(gx, a.S), dim3(WM_NW * 64), lds, s, a);
    return hipGetLastError();
}

bool wx_mid_shape(int wt, int x_dt, int64_t M, int64_t N) {
    return wt == WX_Q4 && x_dt != DT_F32 && M > 16 && M <= 64 && N % 8 == 0;
}
bool wx_mid_supported(const WxCall &c) {
    return wx_mid_shape(c.wt, c.x_dt, c.M, c.N) && (uintptr_t)c.W % 16 == 0 &&
           (uintptr_t)c.X % 16 == 0 && c.ldx % 8 == 0 && c.M * c.ldx < ((int64_t)1 << 30) &&
           (c.K / QK) * c.N * BLOCK_BYTES < ((int64_t)1 << 31);
}

template <int XT>
static hipError_t launch_wx_mid_x(const WxArgs &a, hipStream_t s) {
    if (a.M <= 32) return launch_wx_mid_t<XT, 2>(a, s);
    if (a.M <= 48) return launch_wx_mid_t<XT, 3>(a, s);
    return launch_wx_mid_t<XT, 4>(a, s);
}

// K splits: one workgroup per CU, every wave at least two K steps.
int wx_mid_splits(int64_t K, int64_t N) {
    const int64_t t = ((N + 63) / 64 + 7) / 8 * 8, nks = K / QK;
    int S = 1;
    while (S < WM_SMAX && t * S * 2 <= 256 && nks / (S * 2 * WM_NW) >= 2) S *= 2;
    return S;
}
// The splits' flag words, behind the partials.
size_t wx_mid_flag_bytes(int64_t N, int S) { return S > 1 ? (size_t)((N + 63) / 64) * S * sizeof(uint32_t) : 0; }

// `a.S` and `a.part` as planned (null: K whole).  *reduce: the partials are left to
// wx_reduce_kernel.  Up to 32 rows split 0 sums (M = 24 4096x4096 8.6 against 9.3 us
// with the reduction, 14336x4096 14.6 against 14.7); above, the second launch, which
// spreads the sums over the chip, costs less than split 0's (M = 33 4096x4096 11.5
// against 14.6, M = 64 14336x4096 21.2 against 33.3).
hipError_t launch_wx_mid(WxArgs a, int x_dt, bool *reduce, hipStream_t s) {
    *reduce = a.S > 1;
    if (a.S > 1 && a.M <= 32 && !opt_is("MCQ4_XCD_LOCAL", '0')) {
        a.flags = (uint32_t *)(a.part + (int64_t)a.S * a.M * a.ldp);
        a.spin = split_spin();
        a.foreign = split_foreign_mask();
        *reduce = false;
    }
    return x_dt == DT_BF16 ? launch_wx_mid_x<DT_BF16>(a, s) : launch_wx_mid_x<DT_F16>(a, s);
}

}  // namespace mcq4
