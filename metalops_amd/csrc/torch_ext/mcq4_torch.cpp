// PyTorch-ROCm extension over the C ABI: the binding a metalcore maintainer
// adds in place of the Metal one.  It mirrors matmul_ggml_q4_0_metal
// (native/core_mps.mm:5917-5975, registered as "matmul_ggml_q4_0" at :6938):
// fp16 X [M, K] and uint8 W_blocks [K/32, N, 18] on the GPU, contiguous copies
// made by the callee, Y [M, N] fp16 allocated by the callee, errors as
// RuntimeError (TORCH_CHECK), work enqueued on the current stream without a
// synchronisation.  The split-K workspace is kept per (device, stream), its counters
// zeroed once (every call leaves them zero); a HIP graph's calls have their own.
//
// It also holds the native call path of the Python functions (q4_matmul, q4_grouped,
// int4_matmul, int8_matmul, int4_rmsnorm below): the checks, the output, the
// workspace and the launch of a call whose tensors need no conversion.  Anything
// else -- other types, strides, alignments, empty shapes, an error -- returns None,
// and the Python function goes its own way: it raises what it raises, or converts the
// tensors and calls again (through ctypes from there, 1024x1024 INT4 with strided
// activations took 24.9 us a call, 16.8 so).  A
// decode call of a 4.3 us kernel took 11.5 us of host time through ctypes.
#include <string>
#include <torch/extension.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <c10/core/DeviceGuard.h>

#include <map>
#include <mutex>
#include <utility>

#include "mcq4.h"

namespace {

// The workspaces of one (device, stream).  `eager` serves the calls that run as they are
// made: on one stream they never overlap, and a larger request replaces it through the
// stream-ordered allocator.  `captured` serves the calls recorded into the stream capture
// `capture`: it comes from the graph's memory pool, so its addresses stay the graph's
// for as long as that can be replayed, whatever later calls on the stream ask for, and no
// eager call or other graph works in it while a replay runs on another stream.  Its
// counters are zeroed by a recorded fill kernel (one per graph and size, 4.2 us of a
// replay), as its memory may hold another graph's data by then.  It is kept
// until the next capture on the stream, so a stream holds at most two buffers.
struct Buffers {
    torch::Tensor eager, captured;
    unsigned long long capture = 0;
};
std::mutex g_ws_mu;
std::map<std::pair<int, hipStream_t>, Buffers> g_ws;

torch::Tensor workspace(int device, hipStream_t stream, size_t need) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(stream, &status, &id) != hipSuccess) {   // the null stream beside another capture
        (void)hipGetLastError();
        status = hipStreamCaptureStatusNone;
    }
    const bool capturing = status == hipStreamCaptureStatusActive;
    std::lock_guard<std::mutex> lk(g_ws_mu);
    Buffers &b = g_ws[{device, stream}];
    torch::Tensor &buf = capturing ? b.captured : b.eager;
    if (!buf.defined() || (size_t)buf.numel() < need || (capturing && b.capture != id)) {
        const size_t bytes = std::max<size_t>(need, 1 << 20);
        // Straight from the allocator: through the dispatcher, a call under a tracing or transform
        // mode would leave that mode's tensor, which has no memory, for every later call.
        const torch::Tensor t = at::detail::empty_cuda({(int64_t)bytes}, at::kByte, at::Device(at::kCUDA, (c10::DeviceIndex)device), std::nullopt);
        const int st = mcq4_reset_workspace(t.data_ptr(), bytes, stream);
        TORCH_CHECK(st == MCQ4_OK, "workspace: ", mcq4_last_error());
        buf = t;
        if (capturing) b.capture = id;
    }
    return buf;
}

}  // namespace

torch::Tensor matmul_ggml_q4_0(torch::Tensor X, torch::Tensor W_blocks) {
    TORCH_CHECK(X.is_cuda(), "X must be on a ROCm GPU");
    TORCH_CHECK(W_blocks.is_cuda() && W_blocks.get_device() == X.get_device(),
                "W_blocks must be on X's GPU");
    TORCH_CHECK(X.scalar_type() == torch::kHalf, "X must be float16");
    TORCH_CHECK(W_blocks.scalar_type() == torch::kUInt8, "W_blocks must be uint8");
    TORCH_CHECK(X.dim() == 2 && W_blocks.dim() == 3, "X must be [M, K] and W_blocks [K/32, N, 18]");
    TORCH_CHECK(W_blocks.size(2) == 18, "W_blocks last dim must be 18 (block_q4_0 size)");
    auto x = X.contiguous();
    auto w = W_blocks.contiguous();
    const int64_t M = x.size(0), K = w.size(0) * 32, N = w.size(1);
    TORCH_CHECK(x.size(1) == K, "X K dimension must match W K dimension");
    if (reinterpret_cast<uintptr_t>(x.data_ptr()) % 16) x = x.clone();   // storage offsets
    if (reinterpret_cast<uintptr_t>(w.data_ptr()) % 2) w = w.clone();
    auto Y = torch::empty({M, N}, x.options());
    if (M == 0 || N == 0) return Y;
    if (K == 0) return Y.zero_();
    const c10::DeviceGuard guard(x.device());   // generic: torch labels ROCm devices "cuda"
    hipStream_t stream = c10::hip::getCurrentHIPStream(x.get_device()).stream();
    const size_t need = mcq4_matmul_workspace_bytes(M, K, N);
    torch::Tensor ws;
    if (need) ws = workspace((int)x.get_device(), stream, need);
    const int st = mcq4_matmul_q4_0_f16(x.data_ptr(), K, w.data_ptr<uint8_t>(), Y.data_ptr(), N, M, K, N,
                                        need ? ws.data_ptr() : nullptr, need ? (size_t)ws.numel() : 0,
                                        stream);
    if (st != MCQ4_OK) {
        // A call that failed after some split-K workgroups drew tickets would leave
        // the per-stream workspace's counter area non-zero for the next call: zero
        // it again (a fill kernel on the same stream) before reporting the error.
        const std::string msg = mcq4_last_error();
        if (need) (void)mcq4_reset_workspace(ws.data_ptr(), (size_t)ws.numel(), stream);
        TORCH_CHECK(false, "matmul_ggml_q4_0: ", mcq4_status_string(st), ": ", msg);
    }
    return Y;
}

namespace {

int dtype_code(at::ScalarType t) {
    return t == at::kHalf ? MCQ4_DTYPE_F16 : t == at::kBFloat16 ? MCQ4_DTYPE_BF16 : t == at::kFloat ? MCQ4_DTYPE_F32 : -1;
}
bool at16(const at::Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// A plain tensor (or parameter) on a GPU, or null.
const at::Tensor *gpu_tensor(PyObject *o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}

// Device, stream and workspace of one call.
struct Call {
    c10::DeviceGuard guard;
    int device;
    hipStream_t stream;
    torch::Tensor ws;
    explicit Call(const at::Tensor &x)
        : guard(x.device()), device((int)x.get_device()), stream(c10::hip::getCurrentHIPStream(x.get_device()).stream()) {}
    void *need(size_t n) {
        if (!n) return nullptr;
        ws = workspace(device, stream, n);
        return ws.data_ptr();
    }
    size_t bytes() const { return ws.defined() ? (size_t)ws.numel() : 0; }
    // False after a failed call, its workspace's counters zeroed again.
    bool ok(int st, void *base = nullptr) {
        if (st == MCQ4_OK) return true;
        if (ws.defined()) {
            char *p = base ? (char *)base : (char *)ws.data_ptr();
            (void)mcq4_reset_workspace(p, bytes() - (size_t)(p - (char *)ws.data_ptr()), stream);
        }
        return false;
    }
};

// Rows the kernels take as they are: unit column stride, fp16 16-byte aligned.
bool rows_ok(const at::Tensor &x, int64_t K, bool align16) {
    return x.stride(1) == 1 && x.stride(0) >= K && (!align16 || (x.stride(0) % 8 == 0 && at16(x)));
}
bool blocks_ok(const at::Tensor &w, const at::Tensor &x) {
    return w.device() == x.device() && w.scalar_type() == at::kByte && w.dim() == 3 && w.size(2) == 18 && w.is_contiguous() &&
           reinterpret_cast<uintptr_t>(w.data_ptr()) % 2 == 0;
}

template <typename F>
PyObject *native_call(F body) {
    try {
        at::Tensor y = body();
        if (y.defined()) return THPVariable_Wrap(std::move(y));
    } catch (...) {                              // Python's path meets the same condition and raises it
    }
    PyErr_Clear();
    Py_RETURN_NONE;
}

// q4_matmul(X, W_blocks)
PyObject *q4_matmul(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return native_call([&]() -> at::Tensor {
        const at::Tensor *X = n == 2 ? gpu_tensor(args[0]) : nullptr, *W = X ? gpu_tensor(args[1]) : nullptr;
        if (!W || X->dim() != 2 || !blocks_ok(*W, *X)) return {};
        const int dt = dtype_code(X->scalar_type());
        const int64_t M = X->size(0), K = W->size(0) * 32, N = W->size(1);
        if (dt < 0 || X->size(1) != K || M == 0 || N == 0 || K == 0 || !rows_ok(*X, K, dt == MCQ4_DTYPE_F16)) return {};
        Call c(*X);
        at::Tensor Y = at::empty({M, N}, X->options());
        void *ws = c.need(mcq4_matmul_q4_0_workspace_bytes(M, K, N, dt));
        if (!c.ok(mcq4_matmul_q4_0(X->data_ptr(), dt, X->stride(0), (const uint8_t *)W->data_ptr(), Y.data_ptr(), N, M, K, N, ws,
                                   c.bytes(), c.stream)))
            return {};
        return Y;
    });
}

// int4 / int8: fn(X, W_packed, scales, zeros, group_size, act)
at::Tensor grouped_matmul(PyObject *const *args, Py_ssize_t n, int wb) {
    if (n != 6) return {};
    const at::Tensor *X = gpu_tensor(args[0]), *P = gpu_tensor(args[1]), *S = gpu_tensor(args[2]), *Z = gpu_tensor(args[3]);
    if (!X || !P || !S || !Z || !PyLong_CheckExact(args[4]) || !PyLong_CheckExact(args[5])) return {};
    const long long gs = PyLong_AsLongLong(args[4]), act = PyLong_AsLongLong(args[5]);
    const int dt = dtype_code(X->scalar_type()), sdt = dtype_code(S->scalar_type());
    if (gs <= 0 || dt < 0 || sdt < 0 || (X->dim() != 2 && !(wb == 4 && X->dim() == 3)) || P->dim() != 2 || S->dim() != 2) return {};
    if (act != 0 && (dt != MCQ4_DTYPE_F16 || X->dim() != 2)) return {};
    const int64_t K = P->size(0) * (wb == 4 ? 2 : 1), N = P->size(1), G = (K + gs - 1) / gs;
    if (P->device() != X->device() || S->device() != X->device() || Z->device() != X->device()) return {};
    if ((P->scalar_type() != at::kByte && !(wb == 8 && P->scalar_type() == at::kChar)) || S->size(0) != G || S->size(1) != N ||
        Z->sizes() != S->sizes() || Z->scalar_type() != S->scalar_type())
        return {};
    if (!P->is_contiguous() || !S->is_contiguous() || !Z->is_contiguous() || !at16(*P) || !at16(*S) || !at16(*Z)) return {};
    const int64_t M = X->dim() == 3 ? X->size(0) * X->size(1) : X->size(0);
    if (X->size(-1) != K || M == 0 || N == 0 || K == 0) return {};
    if (X->dim() == 3 ? !(X->is_contiguous() && K % 8 == 0 && at16(*X)) : !rows_ok(*X, K, true)) return {};
    Call c(*X);
    at::Tensor Y = X->dim() == 3 ? at::empty({X->size(0), X->size(1), N}, X->options()) : at::empty({M, N}, X->options());
    const int64_t ldx = X->dim() == 3 ? K : X->stride(0);
    void *ws = c.need(wb == 4 ? mcq4_matmul_int4_best_workspace_bytes(M, K, N, gs, dt) : mcq4_matmul_int8_best_workspace_bytes(M, K, N, gs, dt));
    int st;
    if (wb == 8)
        st = mcq4_matmul_int8(X->data_ptr(), dt, ldx, (const int8_t *)P->data_ptr(), S->data_ptr(), Z->data_ptr(), sdt, Y.data_ptr(), N, M,
                              K, N, gs, ws, c.bytes(), c.stream);
    else
        st = (act == 1 ? mcq4_matmul_int4_silu : act == 2 ? mcq4_matmul_int4_gelu : mcq4_matmul_int4)(
            X->data_ptr(), dt, ldx, (const uint8_t *)P->data_ptr(), S->data_ptr(), Z->data_ptr(), sdt, Y.data_ptr(), N, M, K, N, gs, ws,
            c.bytes(), c.stream);
    if (!c.ok(st)) return {};
    return Y;
}
PyObject *int4_matmul(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return native_call([&] { return grouped_matmul(args, n, 4); });
}
PyObject *int8_matmul(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return native_call([&] { return grouped_matmul(args, n, 8); });
}

// int4_rmsnorm(X, W_norm, W_packed, scales, zeros, eps, group_size)
PyObject *int4_rmsnorm(PyObject *, PyObject *const *args, Py_ssize_t n) {
    return native_call([&]() -> at::Tensor {
        if (n != 7 || !PyFloat_CheckExact(args[5]) || !PyLong_CheckExact(args[6])) return {};
        const at::Tensor *X = gpu_tensor(args[0]), *w = gpu_tensor(args[1]), *P = gpu_tensor(args[2]), *S = gpu_tensor(args[3]),
                         *Z = gpu_tensor(args[4]);
        if (!X || !w || !P || !S || !Z) return {};
        const float eps = (float)PyFloat_AsDouble(args[5]);
        const long long gs = PyLong_AsLongLong(args[6]);
        const int sdt = dtype_code(S->scalar_type());
        if (gs <= 0 || sdt < 0 || X->dim() != 2 || P->dim() != 2 || S->dim() != 2 || w->dim() != 1) return {};
        const int64_t M = X->size(0), K = P->size(0) * 2, N = P->size(1), G = (K + gs - 1) / gs;
        for (const at::Tensor *t : {w, P, S, Z})
            if (t->device() != X->device() || !t->is_contiguous()) return {};
        if (X->scalar_type() != at::kHalf || w->scalar_type() != at::kHalf || P->scalar_type() != at::kByte || X->size(1) != K ||
            w->size(0) != K || S->size(0) != G || S->size(1) != N || Z->sizes() != S->sizes() || Z->scalar_type() != S->scalar_type())
            return {};
        if (M == 0 || N == 0 || K == 0 || !at16(*P) || !at16(*S) || !at16(*Z) || X->stride(1) != 1 || X->stride(0) < K ||
            reinterpret_cast<uintptr_t>(X->data_ptr()) % 2)
            return {};
        Call c(*X);
        at::Tensor Y = at::empty({M, N}, X->options());
        const uintptr_t ws = (uintptr_t)c.need(mcq4_fused_rmsnorm_linear_int4_workspace_bytes(M, K, N, gs) + 256);
        void *base = (void *)((ws + 255) / 256 * 256);
        if (!c.ok(mcq4_fused_rmsnorm_linear_int4(X->data_ptr(), X->stride(0), w->data_ptr(), eps, (const uint8_t *)P->data_ptr(),
                                                 S->data_ptr(), Z->data_ptr(), sdt, Y.data_ptr(), N, M, K, N, gs, base,
                                                 c.bytes() - ((uintptr_t)base - ws), c.stream),
                  base))
            return {};
        return Y;
    });
}

// q4_grouped(X, [W, ...]): one fp16 row, up to four weights of one shape, N % 16 == 0.
PyObject *q4_grouped(PyObject *, PyObject *const *args, Py_ssize_t n) {
    at::Tensor Y[4];
    Py_ssize_t count = 0;
    try {
        const at::Tensor *X = n == 2 ? gpu_tensor(args[0]) : nullptr;
        if (X && PyList_CheckExact(args[1])) count = PyList_GET_SIZE(args[1]);
        if (!X || count < 1 || count > 4 || X->dim() != 2 || X->size(0) != 1 || X->scalar_type() != at::kHalf) Py_RETURN_NONE;
        const uint8_t *wp[4];
        void *yp[4];
        int64_t K = 0, N = 0;
        for (Py_ssize_t i = 0; i < count; ++i) {
            const at::Tensor *W = gpu_tensor(PyList_GET_ITEM(args[1], i));
            if (!W || !blocks_ok(*W, *X) || !at16(*W)) Py_RETURN_NONE;
            if (i == 0) { K = W->size(0) * 32; N = W->size(1); }
            if (W->size(0) * 32 != K || W->size(1) != N) Py_RETURN_NONE;
            wp[i] = (const uint8_t *)W->data_ptr();
        }
        if (K == 0 || N == 0 || N % 16 || X->size(1) != K || !rows_ok(*X, K, true)) Py_RETURN_NONE;
        Call c(*X);
        for (Py_ssize_t i = 0; i < count; ++i) {
            Y[i] = at::empty({1, N}, X->options());
            yp[i] = Y[i].data_ptr();
        }
        void *ws = c.need(mcq4_matmul_workspace_bytes(1, K, N));
        if (!c.ok(mcq4_matmul_q4_0_f16_grouped(X->data_ptr(), X->stride(0), (int)count, wp, yp, N, 1, K, N, ws, c.bytes(), c.stream)))
            Py_RETURN_NONE;
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    PyObject *out = PyList_New(count);
    for (Py_ssize_t i = 0; out && i < count; ++i) PyList_SET_ITEM(out, i, THPVariable_Wrap(std::move(Y[i])));
    return out;
}

// workspace(device index, stream, bytes): the same buffers for the Python path.
torch::Tensor py_workspace(int device, int64_t stream, int64_t bytes) {
    return workspace(device, (hipStream_t)(intptr_t)stream, (size_t)bytes);
}

PyMethodDef g_methods[] = {
    {"q4_matmul", (PyCFunction)(void (*)(void))q4_matmul, METH_FASTCALL, nullptr},
    {"q4_grouped", (PyCFunction)(void (*)(void))q4_grouped, METH_FASTCALL, nullptr},
    {"int4_matmul", (PyCFunction)(void (*)(void))int4_matmul, METH_FASTCALL, nullptr},
    {"int8_matmul", (PyCFunction)(void (*)(void))int8_matmul, METH_FASTCALL, nullptr},
    {"int4_rmsnorm", (PyCFunction)(void (*)(void))int4_rmsnorm, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("matmul_ggml_q4_0", &matmul_ggml_q4_0, "GGML block_q4_0 matmul (gfx950 HIP kernels)");
    m.def("workspace", &py_workspace);
    if (PyModule_AddFunctions(m.ptr(), g_methods) != 0) throw pybind11::error_already_set();
}
