// C ABI of the gfx950 q4_0 path: argument validation, status codes and
// dispatch to the kernel launchers.  No allocation, no exceptions; everything
// is enqueued on the caller's stream.
//
// Reference boundary replaced: metalcore's pybind11 binding
// matmul_ggml_q4_0_metal (native/core_mps.mm:5917-5975): shape/dtype checks
// (core_mps.mm:5923-5938) become status codes, the Metal encode on the current
// MPS stream (core_mps.mm:5947-5969) becomes a launch on the given HIP stream.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <stdarg.h>
#include <stdio.h>

#include "../../include/mcq4.h"
#include "q4_prefill.h"
#include "wx_common.h"

namespace mcq4 {
hipError_t launch_quantize(bool llama_rule, const float *W, int64_t ldw, int nb, int N,
                           uint8_t *out, hipStream_t s);
hipError_t launch_dequant(const uint8_t *blocks, int nb, int N, void *out, int64_t ldo, int out_dt, hipStream_t s);
size_t skinny_workspace_bytes(int64_t M, int64_t K, int64_t N);
hipError_t launch_skinny(const _Float16 *X, int64_t ldx, const uint8_t *W, _Float16 *Y,
                         int64_t ldy, int M, int K, int N, void *ws, hipStream_t s);
size_t gemm_workspace_bytes(int64_t M, int64_t K, int64_t N);
hipError_t launch_gemm(const _Float16 *X, int64_t ldx, const uint8_t *W, _Float16 *Y,
                       int64_t ldy, int M, int K, int N, void *ws, hipStream_t s);
bool gemm2_supported(const _Float16 *X, int64_t ldx, const uint8_t *W, int64_t K, int64_t N);
hipError_t launch_gemm2(const _Float16 *X, int64_t ldx, const uint8_t *W, _Float16 *Y,
                        int64_t ldy, int M, int K, int N, hipStream_t s);
hipError_t launch_quantize_typed(int w_dtype, const void *W, int64_t ldw, int nb, int N,
                                 uint8_t *out, hipStream_t s);
hipError_t launch_zero_counters(void *ws, hipStream_t s);
size_t gemm7_workspace_bytes(int64_t M, int64_t K, int64_t N);
bool gemm7_supported(const _Float16 *X, int64_t ldx, const uint8_t *W, int64_t M, int64_t K, int64_t N);
hipError_t launch_gemm7(const _Float16 *X, int64_t ldx, const uint8_t *W, _Float16 *Y,
                        int64_t ldy, int M, int K, int N, int x_dt, void *ws, hipStream_t s);
hipError_t q4_gemvm_split_fallbacks(uint64_t *count, bool reset);
hipError_t q4_gemm6_split_fallbacks(uint64_t *count, bool reset);
hipError_t i4_gemv_split_fallbacks(uint64_t *count, bool reset);
hipError_t i4_gemv1_split_fallbacks(uint64_t *count, bool reset);
hipError_t i4_gemm6_split_fallbacks(uint64_t *count, bool reset);
size_t gemv_span_bf16_workspace_bytes(int64_t M, int64_t K, int64_t N);
hipError_t launch_gemv_span_bf16(const void *X, int64_t ldx, const uint8_t *W, void *Y, int64_t ldy, int64_t M, int64_t K,
                                 int64_t N, void *ws, size_t ws_bytes, bool *done, hipStream_t s);
hipError_t q4_gemv_span_split_fallbacks(uint64_t *count, bool reset);
hipError_t q4_gemm8_split_fallbacks(uint64_t *count, bool reset);
hipError_t wx_mid_split_fallbacks(uint64_t *count, bool reset);
bool wx_mid_supported(const WxCall &c);
bool gemv_dma_supported(const _Float16 *X, const uint8_t *W, int64_t K, int64_t N);
hipError_t launch_gemv_dma_group(const _Float16 *X, const uint8_t *const *W, _Float16 *const *Y, int count,
                                 int K, int N, int *n_done, hipStream_t s);
}  // namespace mcq4

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int hip_status(hipError_t e, const char *what) {
    if (e == hipSuccess) return MCQ4_OK;
    return fail(MCQ4_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

constexpr int64_t kMaxBlocksK = 65535;        // grid.y limit of the conversion kernels
constexpr int64_t kMaxDim = (int64_t)1 << 30;  // keeps 32-bit lane offsets safe

bool aligned(const void *p, uintptr_t a) { return ((uintptr_t)p % a) == 0; }

// Prefill kernel choice (M > 64).  When N % 8 == 0 and the pointers are
// 16-byte aligned: the few-tile GEMM (q4_gemm8, N % 128 == 0) when its plan is
// one round of workgroups, the 256 x 256-tile GEMM (q4_gemm7) on grids that
// nearly fill the CUs, else the 128 x 256-tile LDS-staged GEMM with two waves per
// SIMD (q4_gemm6).  Otherwise the kernel without alignment needs (wx_gemm).
// fp16 on short K, unless N % 128 == 0 and aligned: the register-staged q4_gemm.
// MCQ4_GEMM_PATH=sync|async|6|7|8 forces one kernel (tests; sync and async are
// the fp16 kernels q4_gemm and q4_gemm2).
enum class Prefill { Sync, Async2, Staged6, Wide7, Few8, Any };
Prefill prefill_kernel(const _Float16 *X, int64_t ldx, const uint8_t *W, int64_t M, int64_t K,
                       int64_t N, bool f16) {
    const bool ok2 = mcq4::gemm2_supported(X, ldx, W, K, N);
    const bool ok6 = mcq4::gemm6_supported(X, ldx, W, M, K, N);
    if (const char *env = mcq4::opt("MCQ4_GEMM_PATH")) {
        if (env[0] == 's') return Prefill::Sync;
        if (env[0] == 'a' && ok2) return Prefill::Async2;
        if (env[0] == '6' && ok6) return Prefill::Staged6;
        if (env[0] == '7' && mcq4::gemm7_supported(X, ldx, W, M, K, N)) return Prefill::Wide7;
        if (env[0] == '8' && mcq4::gemm8_supported(X, ldx, W, M, K, N)) return Prefill::Few8;
    }
    // Short K: filling wx_gemm's register ring and two LDS slots and summing its phases takes
    // about 10 us whatever K is, q4_gemm6's stages about 8; q4_gemm starts sooner, takes
    // longer per K step and needs more rounds of workgroups on wide outputs.  us, q4_gemm /
    // q4_gemm6: 300x32x1032 5.5 / 7.7, x128 8.1 / 8.9, x160 9.0 / 9.4, 2048x32x4104 16.3 / 11.3; /
    // wx_gemm: 300x32x1001 5.4 / 10.7, x256 11.6 / 13.1, x384 15.2 / 14.9; 512x256x8193 13.5 /
    // 14.8, 1024x128x6001 11.2 / 13.5, 300x192x14335 15.3 / 13.8; 2048x32x8193 40.3 / 32.3.
    const int64_t t6 = ((M + 127) / 128) * ((N + 255) / 256);
    if (f16 && (ok6 ? N % 128 != 0 && K < 160 && t6 <= 128 : K < (t6 <= 144 ? 384 : t6 <= 288 ? 160 : 0)))
        return Prefill::Sync;
    // Measured (us per launch, `python bench.py --part prefill-routing`, one box;
    // default / q4_gemm6 / q4_gemm7 / q4_gemm8 forced):
    //   M=512 11008x4096 55.8 / 59.5 / 64.1 / 56.5, 4096x4096 29.3 / 31.7 / 35.6 / 29.3
    //   M=768 4096x4096 35.1 / 43.9 / 43.6 / 35.0; M=1024 4096x4096 40.8 / 50.2 / 53.2 / 41.0
    //   M=256 4096x14336 39.7 / 46.7 / 49.1 / 39.7
    //   M=1024 4096x11008 96.1 / 109.0 / 96.4 / 116.1; M=768 4096x14336 94.7 / 107.9 / 94.8 / 114.8
    //   M=1280 4096x8192 92.2 / 106.2 / 92.4 / 111.6
    //   M=640 4096x11008 69.9 / 69.1 / 85.8 / 75.7; M=1536 4096x4096 63.3 / 63.2 / 65.3 / 72.6
    //   M=256 11008x4096 38.0 / 38.6 / 43.6 / 41.1; M=2048 4096x4096 75.0 / 75.1 / 81.0 / 81.5
    // The few-tile GEMM (128 x 128 tiles, eight waves, K split four ways
    // inside the workgroup and at most twice across) wins when its plan is one
    // round of 192..256 workgroups, and loses with more rounds or a half-empty
    // grid.  The 256 x 256-tile GEMM (one wave per SIMD, half the dequant per
    // MFMA) wins from 160 tiles, or from 96 on long K where two K splits and
    // their reduction cost little; the 128 x 256-tile q4_gemm6 below that.
    if (ok6 && mcq4::gemm8_supported(X, ldx, W, M, K, N)) {
        const int g8 = mcq4::gemm8_workgroups(M, K, N);
        if (g8 >= 192 && g8 <= 256) return Prefill::Few8;
    }
    if (ok6 && mcq4::gemm7_supported(X, ldx, W, M, K, N)) {
        const int64_t t7 = ((M + 255) / 256) * ((N + 255) / 256);
        if (t7 >= 160 || (t7 >= 96 && K >= 8192)) return Prefill::Wide7;
    }
    if (ok6) return Prefill::Staged6;
    return Prefill::Any;
}

// The most any of the aligned prefill kernels asks for.
size_t prefill_ws_bytes(int64_t M, int64_t K, int64_t N) {
    return std::max({mcq4::gemm6_workspace_bytes(M, K, N), mcq4::gemm7_workspace_bytes(M, K, N),
                     mcq4::gemm8_workspace_bytes(M, K, N)});
}

// Switches (tests) that leave 17..64 fp16 rows to the decode kernels.
bool decode_switch() {
    return mcq4::opt("MCQ4_GEMVM_SPLIT") || mcq4::opt("MCQ4_GEMV_PATH") || mcq4::opt("MCQ4_DECODE_PATH");
}

// 33..64 fp16 rows that the strip kernels keep (8 columns: q4_skinny): at most 4096 columns in
// strips of 16 are one round of workgroups, and wx_mid's K split and its reduction
// launch cost more than they save on short K.  us, strips / wx_mid: M=48 1024x528 5.7 / 8.7, M=33 2048x1040
// 8.3 / 8.6, M=64 1536x1040 9.6 / 9.8, M=33 128x8 3.8 / 4.7; M=48 3072x528 11.1 / 9.4, M=64
// 2048x512 10.2 / 9.3, M=48 1024x4112 9.2 / 9.3.
bool strip_rows(int64_t M, int64_t K, int64_t N) {
    return ((N % 16 == 0 && N <= 4096) || N == 8) && K < (M <= 48 ? 2560 : 2048);
}

// 17..64 fp16 rows of the kernel between the decode and the prefill ones (wx_mid).  Up to 32
// rows from K = 4096 on (us, q4_gemvm / wx_mid: M=32 4096x14336 18.4 / 13.5, M=17 4096x4096
// 9.3 / 8.8; M=32 2048x4096 7.3 / 7.6, M=17 1024x4096 4.7 / 6.4).  Above, where the strips do
// not keep them, up to 16384 columns (256 tiles of 64, one per CU) at any K; in further
// rounds of tiles once K is long enough for the weights' bytes to count, and above 56 rows
// not where the few-tile prefill kernel (q4_gemm8) has one round of workgroups, up to K = 4096.
// us, prefill kernel / wx_mid: M=64 4096x14336 29.3 / 17.6, 256x16384 10.7 / 6.3, 256x17920
// 10.7 / 10.1; M=48 128x17920 8.8 / 8.6, 128x128256 24.4 / 29.2, 512x128256 39.9 / 40.7; M=64
// 512x32000 11.9 / 13.0, 3072x32000 30.8 / 32.8, 4096x32000 39.7 / 36.5, 3072x49152 70.6 / 48.0.
bool mid_rows(int64_t M, int64_t K, int64_t N) {
    if (M <= 16 || M > 64) return false;
    if (M <= 32) return K >= 4096;
    if (strip_rows(M, K, N)) return false;
    if (N <= 16384) return true;
    const int64_t g8 = N % 128 == 0 ? mcq4::gemm8_workgroups(M, K, N) : 0;
    return K >= (N <= 65536 ? 256 : 512) && !(M > 56 && K < 4096 && g8 >= 192 && g8 <= 256);
}

// Up to 64 fp16 rows of weights the strip kernels do not take (odd column counts or addresses)
// that run wx_gemv / wx_skinny, LDS sums over 16 or 8 waves instead of q4_skinny's 4, with the
// same arithmetic (weights rounded to fp16): more than 4096 columns from K = 4096 on, where
// q4_skinny has a second round of workgroups; with fewer, once K outweighs the longer sums.
// us, q4_skinny / wx: M=1 4096x4097 9.4 / 8.6, 4096x8193 14.7 / 10.5, M=16 4096x4097 13.9 / 11.7,
// M=64 4096x8193 43.7 / 28.9; up to 4096 columns M=1 4096x1001 6.7 / 5.9, M=8 4096x33 7.1 / 7.5,
// 5120x33 8.7 / 8.5, M=16 4096x3001 9.1 / 10.0, 8192x33 13.2 / 14.0, 10240x33 16.7 / 16.2, M=17
// 4096x3001 9.7 / 11.0, 5120x3001 12.0 / 11.5, M=33 4096x4095 13.7 / 14.2, M=48 4096x3001 16.2 / 15.4.
bool loose_rows(int64_t M, int64_t K, int64_t N) {
    if (M > 64 || K < 4096) return false;
    return N > 4096 || M <= 4 || M > 40 || K >= (M > 8 && M <= 16 ? 10240 : 5120);
}

int check_kn(int64_t K, int64_t N) {
    if (K <= 0 || N <= 0) return fail(MCQ4_ERR_SHAPE, "K (%lld) and N (%lld) must be positive",
                                      (long long)K, (long long)N);
    if (K % 32 != 0) return fail(MCQ4_ERR_SHAPE, "K (%lld) must be divisible by 32", (long long)K);
    if (K / 32 > kMaxBlocksK || N > kMaxDim || (K / 32) * N * 18 > ((int64_t)1 << 40))
        return fail(MCQ4_ERR_SHAPE, "shape K=%lld N=%lld exceeds the supported size",
                    (long long)K, (long long)N);
    return MCQ4_OK;
}

// Scratch of the allocation-free matmul entry point: one split-K workspace per
// GPU in the library's own device memory (zero at load; every completed call
// leaves its counter area zero again).  Host code uses only the per-device
// address from hipGetSymbolAddress, never the array's name.  16 MiB of partials
// hold every decode shape's split-K plan (1.25 MiB at M = 16..32, K = 14336) and
// prefill plans up to M = 64 at K = 14336; larger split-K plans are rejected.
// The array is part of the library image, so every GPU the library is loaded on
// holds it (16.25 MiB) whether or not the entry point is called.
constexpr size_t kNoAllocScratchBytes = mcq4::COUNTER_BYTES + ((size_t)16 << 20);
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];
constexpr int kMaxDevices = 64;
std::atomic<void *> g_scratch[kMaxDevices];
std::atomic<bool> g_scratch_dirty[kMaxDevices];   // a failed call may have left counters set
std::mutex g_scratch_mu;

// The current device's scratch address, resolved once per device.
int scratch_ptr(void **out, int *dev_out) {
    int dev = 0;
    if (hipError_t e = hipGetDevice(&dev)) return hip_status(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail(MCQ4_ERR_INVALID_ARG, "device %d out of range", dev);
    void *p = g_scratch[dev].load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        p = g_scratch[dev].load(std::memory_order_acquire);
        if (!p) {
            if (hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)))
                return hip_status(e, "hipGetSymbolAddress(scratch)");
            if (!p) return fail(MCQ4_ERR_HIP, "hipGetSymbolAddress(scratch) returned null");
            g_scratch[dev].store(p, std::memory_order_release);
        }
    }
    *out = p;
    *dev_out = dev;
    return MCQ4_OK;
}

}  // namespace

namespace mcq4 {
int set_error(int code, const char *msg) {
    snprintf(g_err, sizeof(g_err), "%s", msg);
    return code;
}
}  // namespace mcq4

extern "C" {

int mcq4_version(void) { return 1 * 10000 + 1 * 100 + 0; }

const char *mcq4_status_string(int status) {
    switch (status) {
        case MCQ4_OK: return "ok";
        case MCQ4_ERR_INVALID_ARG: return "invalid argument";
        case MCQ4_ERR_SHAPE: return "unsupported shape";
        case MCQ4_ERR_ALIGNMENT: return "misaligned pointer or leading dimension";
        case MCQ4_ERR_WORKSPACE: return "workspace missing or too small";
        case MCQ4_ERR_HIP: return "HIP runtime error";
        default: return "unknown status";
    }
}

const char *mcq4_last_error(void) { return g_err; }

static int quantize_common(bool llama, const float *W, int64_t ldw, int64_t K, int64_t N,
                           uint8_t *blocks, void *stream) {
    g_err[0] = 0;
    if (!W || !blocks) return fail(MCQ4_ERR_INVALID_ARG, "null pointer");
    if (int st = check_kn(K, N)) return st;
    if (ldw < N) return fail(MCQ4_ERR_SHAPE, "ldw (%lld) < N (%lld)", (long long)ldw, (long long)N);
    if (!aligned(W, 4)) return fail(MCQ4_ERR_ALIGNMENT, "W must be 4-byte aligned");
    if (!aligned(blocks, 2)) return fail(MCQ4_ERR_ALIGNMENT, "blocks must be 2-byte aligned");
    return hip_status(mcq4::launch_quantize(llama, W, ldw, (int)(K / 32), (int)N, blocks,
                                            (hipStream_t)stream),
                      "quantize launch");
}

int mcq4_quantize_q4_0(const float *W, int64_t ldw, int64_t K, int64_t N, uint8_t *blocks,
                       void *stream) {
    return quantize_common(false, W, ldw, K, N, blocks, stream);
}

int mcq4_quantize_q4_0_typed(const void *W, int w_dtype, int64_t ldw, int64_t K, int64_t N,
                             uint8_t *blocks, void *stream) {
    g_err[0] = 0;
    if (!W || !blocks) return fail(MCQ4_ERR_INVALID_ARG, "null pointer");
    if (w_dtype != MCQ4_DTYPE_F32 && w_dtype != MCQ4_DTYPE_F16 && w_dtype != MCQ4_DTYPE_BF16)
        return fail(MCQ4_ERR_INVALID_ARG, "w_dtype must be MCQ4_DTYPE_F32, F16 or BF16");
    if (int st = check_kn(K, N)) return st;
    if (ldw < N) return fail(MCQ4_ERR_SHAPE, "ldw (%lld) < N (%lld)", (long long)ldw, (long long)N);
    if (!aligned(W, w_dtype == MCQ4_DTYPE_F32 ? 4 : 2))
        return fail(MCQ4_ERR_ALIGNMENT, "W is misaligned for its dtype");
    if (!aligned(blocks, 2)) return fail(MCQ4_ERR_ALIGNMENT, "blocks must be 2-byte aligned");
    return hip_status(mcq4::launch_quantize_typed(w_dtype, W, ldw, (int)(K / 32), (int)N, blocks,
                                                  (hipStream_t)stream),
                      "quantize launch");
}

int mcq4_quantize_q4_0_llama(const float *W, int64_t ldw, int64_t K, int64_t N,
                             uint8_t *blocks, void *stream) {
    return quantize_common(true, W, ldw, K, N, blocks, stream);
}

static int dequantize_common(const uint8_t *blocks, int64_t K, int64_t N, void *out, int64_t ldo, int out_dtype,
                             void *stream) {
    if (!blocks || !out) return fail(MCQ4_ERR_INVALID_ARG, "null pointer");
    if (int st = check_kn(K, N)) return st;
    if (ldo < N) return fail(MCQ4_ERR_SHAPE, "ldo (%lld) < N (%lld)", (long long)ldo, (long long)N);
    if (!aligned(blocks, 2)) return fail(MCQ4_ERR_ALIGNMENT, "blocks must be 2-byte aligned");
    if (!aligned(out, out_dtype == MCQ4_DTYPE_F32 ? 4 : 2))
        return fail(MCQ4_ERR_ALIGNMENT, "out is misaligned for its dtype");
    return hip_status(mcq4::launch_dequant(blocks, (int)(K / 32), (int)N, out, ldo, out_dtype, (hipStream_t)stream),
                      "dequantize launch");
}

int mcq4_dequantize_q4_0(const uint8_t *blocks, int64_t K, int64_t N, void *out, int64_t ldo,
                         int out_dtype, void *stream) {
    g_err[0] = 0;
    if (!blocks || !out) return fail(MCQ4_ERR_INVALID_ARG, "null pointer");
    if (out_dtype != MCQ4_DTYPE_F32 && out_dtype != MCQ4_DTYPE_F16)
        return fail(MCQ4_ERR_INVALID_ARG, "out_dtype must be MCQ4_DTYPE_F32 or MCQ4_DTYPE_F16");
    return dequantize_common(blocks, K, N, out, ldo, out_dtype, stream);
}

int mcq4_dequantize_q4_0_bf16(const uint8_t *blocks, int64_t K, int64_t N, void *out, int64_t ldo, void *stream) {
    g_err[0] = 0;
    return dequantize_common(blocks, K, N, out, ldo, MCQ4_DTYPE_BF16, stream);
}

// What mcq4_matmul_q4_0_f16 cannot do without: an upper bound over the kernels that a shape
// can reach, whatever the pointers' alignment.  The wx kernels need none, nor does
// q4_gemm at the K it is chosen for.
static size_t required_ws_bytes(int64_t M, int64_t K, int64_t N) {
    if (M <= 0 || K <= 0 || N <= 0 || K % 32) return 0;
    size_t need = M <= 64 ? mcq4::skinny_workspace_bytes(M, K, N) : 0;
    if (M > 64 || (M > 32 && (N > 16384 || decode_switch()))) {
        if (N % 8 == 0) need = std::max(need, prefill_ws_bytes(M, K, N));
        const char *path = mcq4::opt("MCQ4_GEMM_PATH");
        if (path && path[0] == 's') need = std::max(need, mcq4::gemm_workspace_bytes(M, K, N));
    }
    return need;
}

size_t mcq4_matmul_workspace_bytes(int64_t M, int64_t K, int64_t N) {
    const size_t need = required_ws_bytes(M, K, N);
    // wx splits K only where the workspace covers it.
    return M > 16 && K > 0 && N > 0 && K % 32 == 0 ? std::max(need, mcq4::wx_workspace_bytes(mcq4::WX_Q4, mcq4::DT_F16, M, K, N)) : need;
}

size_t mcq4_matmul_q4_0_workspace_bytes(int64_t M, int64_t K, int64_t N, int x_dtype) {
    if (x_dtype == MCQ4_DTYPE_F16) return mcq4_matmul_workspace_bytes(M, K, N);
    if (M <= 0 || K <= 0 || N <= 0 || K % 32) return 0;
    const size_t any = mcq4::wx_workspace_bytes(mcq4::WX_Q4, x_dtype, M, K, N);
    if (x_dtype != MCQ4_DTYPE_BF16) return any;
    return std::max(any, M > 64 ? prefill_ws_bytes(M, K, N) : mcq4::gemv_span_bf16_workspace_bytes(M, K, N));
}

int mcq4_matmul_q4_0_f16(const void *X, int64_t ldx, const uint8_t *W, void *Y, int64_t ldy,
                         int64_t M, int64_t K, int64_t N, void *workspace,
                         size_t workspace_bytes, void *stream) {
    g_err[0] = 0;
    if (!X || !W || !Y) return fail(MCQ4_ERR_INVALID_ARG, "null pointer");
    if (M <= 0) return fail(MCQ4_ERR_SHAPE, "M (%lld) must be positive", (long long)M);
    if (int st = check_kn(K, N)) return st;
    if (M > kMaxDim) return fail(MCQ4_ERR_SHAPE, "M (%lld) too large", (long long)M);
    if (ldx < K) return fail(MCQ4_ERR_SHAPE, "ldx (%lld) < K (%lld)", (long long)ldx, (long long)K);
    if (ldy < N) return fail(MCQ4_ERR_SHAPE, "ldy (%lld) < N (%lld)", (long long)ldy, (long long)N);
    if (!aligned(X, 16) || ldx % 8)
        return fail(MCQ4_ERR_ALIGNMENT, "X must be 16-byte aligned with ldx %% 8 == 0");
    if (!aligned(W, 2)) return fail(MCQ4_ERR_ALIGNMENT, "W must be 2-byte aligned");
    if (!aligned(Y, 2)) return fail(MCQ4_ERR_ALIGNMENT, "Y must be 2-byte aligned");
    const size_t need = required_ws_bytes(M, K, N);
    if (need && (!workspace || workspace_bytes < need))
        return fail(MCQ4_ERR_WORKSPACE, "workspace of %zu bytes required, %zu given", need,
                    workspace ? workspace_bytes : (size_t)0);
    if (need && !aligned(workspace, 16))
        return fail(MCQ4_ERR_ALIGNMENT, "workspace must be 16-byte aligned");
    if (!aligned(workspace, 16)) workspace = nullptr;   // optional from here on: K stays whole
    hipError_t e;
    const mcq4::WxCall wx = {mcq4::WX_Q4, mcq4::DT_F16, 0, mcq4::ACT_NONE, X, ldx, W, nullptr, nullptr, Y, ldy, M, K, N, 32};
    if (mid_rows(M, K, N) && mcq4::wx_mid_supported(wx) && !decode_switch())
        return hip_status(mcq4::launch_wx(wx, workspace, workspace_bytes, (hipStream_t)stream), "matmul launch");
    if (loose_rows(M, K, N) && !(N % 8 == 0 && aligned(W, 16)) && !decode_switch() &&
        mcq4::wx_workspace_bytes(mcq4::WX_Q4, mcq4::DT_F16, M, K, N) <= (workspace ? workspace_bytes : (size_t)0))
        return hip_status(mcq4::launch_wx(wx, workspace, workspace_bytes, (hipStream_t)stream), "matmul launch");
    // 33..64 rows left to here: the strips' shapes, and q4_gemm6 beyond them (by a switch,
    // where N % 128 == 0).
    const bool skinny = M <= 32 || (M <= 64 && (!mcq4::gemm6_supported((const _Float16 *)X, ldx, W, M, K, N) ||
                                                (decode_switch() ? N % 128 != 0 : strip_rows(M, K, N))));
    if (skinny)
        e = mcq4::launch_skinny((const _Float16 *)X, ldx, W, (_Float16 *)Y, ldy, (int)M, (int)K,
                                (int)N, workspace, (hipStream_t)stream);
    else {
        const _Float16 *x = (const _Float16 *)X;
        _Float16 *y = (_Float16 *)Y;
        hipStream_t st = (hipStream_t)stream;
        switch (prefill_kernel(x, ldx, W, M, K, N, true)) {
            case Prefill::Staged6: e = mcq4::launch_gemm6(x, ldx, W, y, ldy, (int)M, (int)K, (int)N, mcq4::DT_F16, workspace, st); break;
            case Prefill::Wide7: e = mcq4::launch_gemm7(x, ldx, W, y, ldy, (int)M, (int)K, (int)N, mcq4::DT_F16, workspace, st); break;
            case Prefill::Few8: e = mcq4::launch_gemm8(x, ldx, W, y, ldy, (int)M, (int)K, (int)N, mcq4::DT_F16, workspace, st); break;
            case Prefill::Async2: e = mcq4::launch_gemm2(x, ldx, W, y, ldy, (int)M, (int)K, (int)N, st); break;
            case Prefill::Any: e = mcq4::launch_wx(wx, workspace, workspace_bytes, st); break;
            default: e = mcq4::launch_gemm(x, ldx, W, y, ldy, (int)M, (int)K, (int)N, workspace, st); break;
        }
    }
    return hip_status(e, "matmul launch");
}

int mcq4_matmul_q4_0_f16_grouped(const void *X, int64_t ldx, int count, const uint8_t *const *W,
                                 void *const *Y, int64_t ldy, int64_t M, int64_t K, int64_t N,
                                 void *workspace, size_t workspace_bytes, void *stream) {
    g_err[0] = 0;
    if (!W || !Y || count < 1) return fail(MCQ4_ERR_INVALID_ARG, "need count >= 1 weights and outputs");
    for (int g = 0; g < count; ++g)
        if (!W[g] || !Y[g]) return fail(MCQ4_ERR_INVALID_ARG, "null weight or output pointer %d", g);
    // The same argument checks as the per-weight calls, whichever path runs.
    if (ldy < N) return fail(MCQ4_ERR_SHAPE, "ldy (%lld) < N (%lld)", (long long)ldy, (long long)N);
    // One launch for M == 1 when every weight takes the M == 1 kernel whole
    // (16-byte aligned, N a multiple of 16) and there are at most 4 of them.
    bool one = M == 1 && count <= 4 && N % 16 == 0 && X && aligned(X, 16) && ldx % 8 == 0 && ldx >= K &&
               K > 0 && K % 32 == 0 && N > 0 && !check_kn(K, N);
    for (int g = 0; one && g < count; ++g)
        one = aligned(Y[g], 2) && mcq4::gemv_dma_supported((const _Float16 *)X, W[g], K, N * count);
    g_err[0] = 0;
    if (!one) {
        for (int g = 0; g < count; ++g)
            if (int st = mcq4_matmul_q4_0_f16(X, ldx, W[g], Y[g], ldy, M, K, N, workspace, workspace_bytes,
                                              stream))
                return st;
        return MCQ4_OK;
    }
    int n_done = 0;
    const hipError_t e = mcq4::launch_gemv_dma_group((const _Float16 *)X, W, (_Float16 *const *)Y, count, (int)K,
                                                     (int)N, &n_done, (hipStream_t)stream);
    return hip_status(e, "grouped matmul launch");
}

int mcq4_matmul_q4_0(const void *X, int x_dtype, int64_t ldx, const uint8_t *W, void *Y,
                     int64_t ldy, int64_t M, int64_t K, int64_t N, void *workspace,
                     size_t workspace_bytes, void *stream) {
    if (x_dtype == MCQ4_DTYPE_F16)
        return mcq4_matmul_q4_0_f16(X, ldx, W, Y, ldy, M, K, N, workspace, workspace_bytes, stream);
    g_err[0] = 0;
    if (x_dtype != MCQ4_DTYPE_F32 && x_dtype != MCQ4_DTYPE_BF16)
        return fail(MCQ4_ERR_INVALID_ARG, "x_dtype must be MCQ4_DTYPE_F32, F16 or BF16");
    if (!X || !W || !Y) return fail(MCQ4_ERR_INVALID_ARG, "null pointer");
    if (M <= 0) return fail(MCQ4_ERR_SHAPE, "M (%lld) must be positive", (long long)M);
    if (int st = check_kn(K, N)) return st;
    if (M > ((int64_t)65535 * 8)) return fail(MCQ4_ERR_SHAPE, "M (%lld) too large", (long long)M);
    if (ldx < K) return fail(MCQ4_ERR_SHAPE, "ldx (%lld) < K (%lld)", (long long)ldx, (long long)K);
    if (ldy < N) return fail(MCQ4_ERR_SHAPE, "ldy (%lld) < N (%lld)", (long long)ldy, (long long)N);
    const uintptr_t al = x_dtype == MCQ4_DTYPE_F32 ? 4 : 2;
    if (!aligned(X, al) || !aligned(Y, al))
        return fail(MCQ4_ERR_ALIGNMENT, "X and Y must be aligned to their dtype");
    if (!aligned(W, 2)) return fail(MCQ4_ERR_ALIGNMENT, "W must be 2-byte aligned");
    if (workspace && !aligned(workspace, 16)) workspace = nullptr;   // optional here: K stays whole
    if (x_dtype == MCQ4_DTYPE_BF16 && M > 64 && aligned(X, 16) && ldx % 8 == 0) {
        // The aligned prefill kernels, where the workspace covers their plans.
        const size_t need = prefill_ws_bytes(M, K, N);
        if (!need || (workspace && workspace_bytes >= need)) {
            const _Float16 *x = (const _Float16 *)X;
            _Float16 *y = (_Float16 *)Y;
            hipStream_t st = (hipStream_t)stream;
            const int m = (int)M, k = (int)K, n = (int)N, dt = mcq4::DT_BF16;
            switch (prefill_kernel(x, ldx, W, M, K, N, false)) {
                case Prefill::Staged6: return hip_status(mcq4::launch_gemm6(x, ldx, W, y, ldy, m, k, n, dt, workspace, st), "matmul launch");
                case Prefill::Wide7: return hip_status(mcq4::launch_gemm7(x, ldx, W, y, ldy, m, k, n, dt, workspace, st), "matmul launch");
                case Prefill::Few8: return hip_status(mcq4::launch_gemm8(x, ldx, W, y, ldy, m, k, n, dt, workspace, st), "matmul launch");
                default: break;
            }
        }
    }
    if (x_dtype == MCQ4_DTYPE_BF16 && M <= 16) {
        bool done = false;
        const hipError_t e = mcq4::launch_gemv_span_bf16(X, ldx, W, Y, ldy, M, K, N, workspace, workspace_bytes, &done, (hipStream_t)stream);
        if (done || e != hipSuccess) return hip_status(e, "matmul launch");
    }
    const mcq4::WxCall c = {mcq4::WX_Q4, x_dtype, 0, mcq4::ACT_NONE, X, ldx, W, nullptr, nullptr, Y, ldy, M, K, N, 32};
    return hip_status(mcq4::launch_wx(c, workspace, workspace_bytes, (hipStream_t)stream), "matmul launch");
}

int mcq4_reset_workspace(void *workspace, size_t workspace_bytes, void *stream) {
    g_err[0] = 0;
    if (!workspace) return fail(MCQ4_ERR_INVALID_ARG, "null workspace");
    if (workspace_bytes < mcq4::COUNTER_BYTES)
        return fail(MCQ4_ERR_WORKSPACE, "workspace of %zu bytes is smaller than its %zu-byte counter area",
                    workspace_bytes, (size_t)mcq4::COUNTER_BYTES);
    if (!aligned(workspace, 16)) return fail(MCQ4_ERR_ALIGNMENT, "workspace must be 16-byte aligned");
    return hip_status(mcq4::launch_zero_counters(workspace, (hipStream_t)stream), "workspace reset launch");
}

int mcq4_split_fallback_count(uint64_t *count, int reset) {
    g_err[0] = 0;
    if (!count) return fail(MCQ4_ERR_INVALID_ARG, "null pointer");
    *count = 0;
    hipError_t (*const readers[])(uint64_t *, bool) = {
        mcq4::q4_gemvm_split_fallbacks, mcq4::q4_gemm6_split_fallbacks, mcq4::i4_gemv_split_fallbacks,
        mcq4::i4_gemv1_split_fallbacks, mcq4::i4_gemm6_split_fallbacks, mcq4::q4_gemv_span_split_fallbacks,
        mcq4::q4_gemm8_split_fallbacks, mcq4::wx_mid_split_fallbacks};
    for (auto rd : readers)
        if (int st = hip_status(rd(count, reset != 0), "split fallback counter")) return st;
    return MCQ4_OK;
}

size_t mcq4_matmul_noalloc_max_workspace_bytes(void) { return kNoAllocScratchBytes; }

int mcq4_matmul_q4_0_f16_noalloc(const void *X, int64_t ldx, const uint8_t *W, void *Y, int64_t ldy,
                                 int64_t M, int64_t K, int64_t N, void *stream) {
    g_err[0] = 0;
    if (M > 0 && K > 0 && N > 0 && K % 32 == 0) {
        const size_t need = required_ws_bytes(M, K, N);
        if (need > kNoAllocScratchBytes)
            return fail(MCQ4_ERR_WORKSPACE,
                        "shape M=%lld K=%lld N=%lld needs a %zu-byte workspace; the allocation-free entry "
                        "point holds at most %zu (use mcq4_matmul_q4_0_f16 with a caller workspace)",
                        (long long)M, (long long)K, (long long)N, need, kNoAllocScratchBytes);
    }
    void *ws = nullptr;
    int dev = 0;
    if (int st = scratch_ptr(&ws, &dev)) return st;
    if (g_scratch_dirty[dev].load(std::memory_order_acquire)) {
        if (int st = hip_status(mcq4::launch_zero_counters(ws, (hipStream_t)stream), "scratch reset launch"))
            return st;
        g_scratch_dirty[dev].store(false, std::memory_order_release);
    }
    const int st = mcq4_matmul_q4_0_f16(X, ldx, W, Y, ldy, M, K, N, ws, kNoAllocScratchBytes, stream);
    // Any failure may follow a launch that drew split-K tickets: the next call
    // zeroes the counter area first.
    if (st != MCQ4_OK) g_scratch_dirty[dev].store(true, std::memory_order_release);
    return st;
}

}  // extern "C"
