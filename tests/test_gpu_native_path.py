"""The native call path of the matmul functions (csrc/torch_ext/mcq4_torch.cpp) around
the kernels: its workspace, what it leaves to the Python functions, and its results
against the ctypes path, bit for bit (the same kernels with the same plans).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _split_call(dev):
    """A call whose K split needs a workspace."""
    import metalops_amd as mo
    from metalops_amd import _lib
    g = torch.Generator(device=dev).manual_seed(3)
    M, K, N = 16, 14336, 4096
    assert _lib.lib.mcq4_matmul_workspace_bytes(M, K, N) > 0
    X = torch.randn(M, K, generator=g, device=dev).half()
    W = mo.quantize_ggml_q4_0_llama(torch.randn(K, N, generator=g, device=dev) * 0.02)
    return lambda: mo.matmul_ggml_q4_0(X, W)


@pytest.mark.parametrize("mode", ["fake", "grad"])
def test_workspace_after_a_tracing_mode(dev, mode):
    """A first call on a stream made under a mode that gives tensors without memory fails, and the
    stream's later calls work."""
    print(f"native path after {mode}", flush=True)
    fn = _split_call(dev)
    ref = fn()
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream(dev)):
        if mode == "fake":
            from torch._subclasses.fake_tensor import FakeTensorMode
            with FakeTensorMode(allow_non_fake_inputs=True), pytest.raises(Exception):
                fn()
        else:
            with pytest.raises(Exception):
                torch.func.grad(lambda x: (fn(), x.sum())[1])(torch.ones(2, device=dev))
        y = fn()
    torch.cuda.synchronize()
    assert torch.equal(y, ref)


def _mods():
    from metalops_amd import int4, quantization
    return quantization, int4


def _without_native(monkeypatch, fn):
    """fn() through ctypes."""
    with monkeypatch.context() as m:
        for mod in _mods():
            m.setattr(mod, "_native", None)
        return fn()


def _bits(y):
    return [t.contiguous().view(torch.uint8) for t in (y if isinstance(y, list) else [y])]


DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


# Every entry; rows of decode, the kernels between and prefill; shapes with and without a K split.
# (silu, gelu and rms are fp16 entries, group takes one fp16 row.)
@pytest.mark.parametrize("op,x,M", [(op, x, M) for op in ("q4", "i4", "i4_3d", "i8") for x in ("f16", "bf16", "f32") for M in (1, 7, 40, 130)]
                         + [(op, "f16", M) for op in ("silu", "gelu", "rms") for M in (1, 7, 40, 130)] + [("group", "f16", 1)])
def test_equals_ctypes_path(dev, monkeypatch, op, x, M):
    import metalops_amd as mo
    print(f"native {op} {x} M={M}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M)
    K, N = 4096, 1040
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    X = rnd(M, K).to(DT[x])
    native = _mods()[0]._native
    if op in ("q4", "group"):
        W = [mo.quantize_ggml_q4_0_llama(rnd(K, N) * 0.02) for _ in range(2)]
        fn = (lambda: mo.matmul_ggml_q4_0(X, W[0])) if op == "q4" else (lambda: mo.matmul_ggml_q4_0_grouped(X, W))
        took = native.q4_matmul(X, W[0]) if op == "q4" else native.q4_grouped(X, W)
    elif op == "i8":
        P = torch.randint(-128, 128, (K, N), generator=g, device=dev, dtype=torch.int8)
        S, Z = (0.002 * rnd(K // 128, N)).to(DT[x]), (3 * rnd(K // 128, N)).to(DT[x])
        fn = lambda: mo.matmul_int8(X, P, S, Z, 128)
        took = native.int8_matmul(X, P, S, Z, 128, 0)
    else:
        P, S, Z = mo.quantize_int4((rnd(K, N) * 0.02).to(DT[x]), 128)
        if op == "rms":
            wn = (1 + 0.1 * rnd(K)).half()
            fn = lambda: mo.fused_rmsnorm_linear_int4(X, wn, P, S, Z, 1e-5, 128)
            took = native.int4_rmsnorm(X, wn, P, S, Z, 1e-5, 128)
        else:
            f = {"silu": mo.matmul_int4_silu, "gelu": mo.matmul_int4_gelu}.get(op, mo.matmul_int4)
            X3 = X[None].expand(1, M, K) if op == "i4_3d" else X
            fn = lambda: f(X3, P, S, Z, 128)
            took = native.int4_matmul(X3, P, S, Z, 128, {"silu": 1, "gelu": 2}.get(op, 0))
    assert took is not None                       # no fall-through: the native path took it
    y, want = fn(), _without_native(monkeypatch, fn)
    for t in (took, y):
        assert all(torch.equal(a, b) for a, b in zip(_bits(t), _bits(want)))
    one = lambda t: t[0] if isinstance(t, list) else t
    assert one(y).shape == one(want).shape and one(y).dtype == one(want).dtype


class _Sub(torch.Tensor):
    pass


def test_leaves_other_calls_to_python(dev, monkeypatch):
    """Strides, offsets, types, devices, subclasses, empty shapes and wrong arguments: the native path returns
    None, and the function gives (or raises) what it does without it."""
    import metalops_amd as mo
    native = _mods()[0]._native
    g = torch.Generator(device=dev).manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    K, N = 256, 64
    W = mo.quantize_ggml_q4_0_llama(rnd(K, N) * 0.02)
    P, S, Z = mo.quantize_int4((rnd(K, N) * 0.02).half(), 32)
    X, wn = rnd(4, K).half(), torch.ones(K, dtype=torch.float16, device=dev)
    wide, flat = rnd(4, 2 * K).half(), rnd(4 * K + 1).half()
    strided = wide[:, ::2]                        # column stride 2
    offset = flat[1:].view(4, K)                  # fp16 rows at an odd element
    w_off = torch.cat([W.reshape(-1)[:1], W.reshape(-1)])[1:].view(W.shape)      # blocks at an odd byte
    w_t = W.transpose(0, 1).contiguous().transpose(0, 1)
    p_t = P.t().contiguous().t()
    calls = {
        "strided": (lambda: native.q4_matmul(strided, W), lambda: mo.matmul_ggml_q4_0(strided, W)),
        "offset": (lambda: native.q4_matmul(offset, W), lambda: mo.matmul_ggml_q4_0(offset, W)),
        "block offset": (lambda: native.q4_matmul(X, w_off), lambda: mo.matmul_ggml_q4_0(X, w_off)),
        "block strides": (lambda: native.q4_matmul(X, w_t), lambda: mo.matmul_ggml_q4_0(X, w_t)),
        "subclass": (lambda: native.q4_matmul(X.as_subclass(_Sub), W), lambda: mo.matmul_ggml_q4_0(X.as_subclass(_Sub), W)),
        "fp64": (lambda: native.q4_matmul(X.double(), W), lambda: mo.matmul_ggml_q4_0(X.double(), W)),
        "no rows": (lambda: native.q4_matmul(X[:0], W), lambda: mo.matmul_ggml_q4_0(X[:0], W)),
        "short K": (lambda: native.q4_matmul(X[:, :64], W), lambda: mo.matmul_ggml_q4_0(X[:, :64], W)),
        "cpu": (lambda: native.q4_matmul(X.cpu(), W), lambda: mo.matmul_ggml_q4_0(X.cpu(), W)),
        "cpu weight": (lambda: native.q4_matmul(X, W.cpu()), lambda: mo.matmul_ggml_q4_0(X, W.cpu())),
        "grouped strides": (lambda: native.q4_grouped(strided[:1], [W, W]), lambda: mo.matmul_ggml_q4_0_grouped(strided[:1], [W, W])),
        "i4 strided": (lambda: native.int4_matmul(strided, P, S, Z, 32, 0), lambda: mo.matmul_int4(strided, P, S, Z, 32)),
        "i4 offset": (lambda: native.int4_matmul(offset, P, S, Z, 32, 0), lambda: mo.matmul_int4(offset, P, S, Z, 32)),
        "i4 weight strides": (lambda: native.int4_matmul(X, p_t, S, Z, 32, 0), lambda: mo.matmul_int4(X, p_t, S, Z, 32)),
        "i4 groups": (lambda: native.int4_matmul(X, P, S, Z, 64, 0), lambda: mo.matmul_int4(X, P, S, Z, 64)),
        "i4 no rows": (lambda: native.int4_matmul(X[:0], P, S, Z, 32, 0), lambda: mo.matmul_int4(X[:0], P, S, Z, 32)),
        "i4 mixed dtypes": (lambda: native.int4_matmul(X, P, S, Z.float(), 32, 0), lambda: mo.matmul_int4(X, P, S, Z.float(), 32)),
        "rms integer eps": (lambda: native.int4_rmsnorm(X, wn, P, S, Z, 1, 32), lambda: mo.fused_rmsnorm_linear_int4(X, wn, P, S, Z, 1, 32)),
        "rms fp32": (lambda: native.int4_rmsnorm(X.float(), wn, P, S, Z, 1e-5, 32),
                     lambda: mo.fused_rmsnorm_linear_int4(X.float(), wn, P, S, Z, 1e-5, 32)),
    }

    def outcome(fn):
        try:
            return _bits(fn())
        except Exception as e:      # the same error on both ways is the point
            return [type(e), str(e)]

    for name, (direct, fn) in calls.items():
        print(f"native path leaves: {name}", flush=True)
        assert direct() is None, name
        a, b = outcome(fn), outcome(lambda: _without_native(monkeypatch, fn))
        assert len(a) == len(b) and all(torch.equal(u, v) if isinstance(u, torch.Tensor) else u == v for u, v in zip(a, b)), (name, a, b)


def test_workspace_grows_and_keeps_its_counters_zero(dev):
    """A larger request replaces the stream's buffer; its counter area is zero before and after calls."""
    native = _mods()[0]._native
    s = torch.cuda.Stream(dev)
    with torch.cuda.stream(s):
        small = native.workspace(dev.index, s.cuda_stream, 1 << 20)
        assert native.workspace(dev.index, s.cuda_stream, 4096).data_ptr() == small.data_ptr()
        large = native.workspace(dev.index, s.cuda_stream, small.numel() + 1)
        assert large.numel() > small.numel() and large.data_ptr() != small.data_ptr()
        assert native.workspace(dev.index, s.cuda_stream, 1 << 20).data_ptr() == large.data_ptr()
        fn = _split_call(dev)
        y = fn()
        z = fn()
        counters = native.workspace(dev.index, s.cuda_stream, 4096)[:256 * 1024].clone()
    torch.cuda.synchronize()
    assert torch.equal(y, z) and not bool(counters.any())


def test_failed_call_zeroes_the_counters(dev):
    """A call that fails after its workspace was fetched (too many rows: refused before any launch) returns
    None and leaves the counter area zero, whatever was there."""
    native = _mods()[0]._native
    M, K, N = 65535 * 8 + 1, 32, 16
    X = torch.zeros(M, K, dtype=torch.float16, device=dev)
    P = torch.zeros(K // 2, N, dtype=torch.uint8, device=dev)
    S = torch.ones(1, N, dtype=torch.float16, device=dev)
    s = torch.cuda.Stream(dev)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        ws = native.workspace(dev.index, s.cuda_stream, 64 << 20)
        ws[:256 * 1024].fill_(1)
        assert native.int4_rmsnorm(X, torch.ones(K, dtype=torch.float16, device=dev), P, S, S, 1e-5, 32) is None
        left = ws[:256 * 1024].clone()
        ws.zero_()
    torch.cuda.synchronize()
    assert not bool(left.any())
