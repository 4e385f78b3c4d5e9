"""Workspaces that the C entry points can do without: one that they cannot use is left
alone, and the call still gives its result.
"""
import pytest
import torch

from oracle import q4_0_ref as Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [(17, 4096, 8192), (65, 8192, 1025), (48, 14336, 4096)])
def test_misaligned_optional_workspace(dev, M, K, N):
    """A buffer that is not 16-byte aligned, where the call requires none but would split K in a larger one:
    the bits of the call without a buffer, nothing written to it."""
    from metalops_amd import _lib
    L = _lib.lib
    print(f"misaligned workspace M={M} K={K} N={N}", flush=True)
    g = torch.Generator().manual_seed(M + N)
    b = torch.from_numpy(Q.quantize_llama_rule((torch.randn(K, N, generator=g) * 0.02).numpy())).to(dev)
    X = torch.randn(M, K, generator=g).half().to(dev)
    stream = torch.cuda.current_stream(dev).cuda_stream
    size = int(L.mcq4_matmul_workspace_bytes(M, K, N))
    assert size > 0

    def call(ws, bytes_):
        Y = torch.full((M, N), float("nan"), dtype=torch.float16, device=dev)
        st = L.mcq4_matmul_q4_0_f16(X.data_ptr(), K, b.data_ptr(), Y.data_ptr(), N, M, K, N, ws, bytes_, stream)
        torch.cuda.synchronize(dev)
        return st, Y

    st, want = call(None, 0)
    assert st == _lib.MCQ4_OK
    buf = torch.full((size + 16,), 0x5A, dtype=torch.uint8, device=dev)
    st, Y = call(buf.data_ptr() + 8, size)
    assert st == _lib.MCQ4_OK and torch.equal(Y.view(torch.int16), want.view(torch.int16))
    assert bool((buf == 0x5A).all())


@pytest.mark.parametrize("M,K,N", [(100, 4096, 4097), (300, 11008, 2049), (48, 14336, 4096), (33, 4096, 1032)])
def test_noalloc_takes_what_needs_no_workspace(dev, M, K, N):
    """Shapes whose kernels can do without a workspace run from the allocation-free entry, with the bits of
    the call with a caller's buffer of the size the query gives."""
    from metalops_amd import _lib
    L = _lib.lib
    print(f"noalloc M={M} K={K} N={N}", flush=True)
    g = torch.Generator().manual_seed(M + N)
    b = torch.randint(0, 256, (K // 32, N, 18), dtype=torch.uint8, generator=g)
    b[:, :, 1] = 0x20
    b, X = b.to(dev), torch.randn(M, K, generator=g).half().to(dev)
    stream = torch.cuda.current_stream(dev).cuda_stream
    size = int(L.mcq4_matmul_workspace_bytes(M, K, N))
    assert size <= int(L.mcq4_matmul_noalloc_max_workspace_bytes())
    ws = torch.zeros(max(size, 16), dtype=torch.uint8, device=dev)
    Y = [torch.full((M, N), float("nan"), dtype=torch.float16, device=dev) for _ in range(2)]
    assert L.mcq4_matmul_q4_0_f16(X.data_ptr(), K, b.data_ptr(), Y[0].data_ptr(), N, M, K, N, ws.data_ptr(), size, stream) == _lib.MCQ4_OK
    assert L.mcq4_matmul_q4_0_f16_noalloc(X.data_ptr(), K, b.data_ptr(), Y[1].data_ptr(), N, M, K, N, stream) == _lib.MCQ4_OK
    torch.cuda.synchronize(dev)
    assert torch.equal(Y[0].view(torch.int16), Y[1].view(torch.int16)) and not bool(Y[0].isnan().any())


@pytest.mark.parametrize("M,K,N", [(33, 4100, 4096), (1, 4100, 4096), (40, 1030, 1000)])
def test_fused_rmsnorm_with_the_required_workspace(dev, M, K, N):
    """The fused RMSNorm + INT4 linear in a buffer that holds the counters and the normalised rows only:
    the product's optional K split is left out, not the call refused.  fp32 sums in another order: each
    output within 2^-10 of itself (two fp16 roundings) and 2 K 2^-24 sum|x w|."""
    from metalops_amd import _lib
    L = _lib.lib
    print(f"fused rmsnorm, smaller workspace M={M} K={K} N={N}", flush=True)
    gs = 128
    g = torch.Generator().manual_seed(M + N)
    X, wn = torch.randn(M, K, generator=g).half(), (1 + 0.1 * torch.randn(K, generator=g)).half()
    P = torch.randint(0, 256, (K // 2, N), dtype=torch.uint8, generator=g)
    S = (0.002 * torch.rand(-(-K // gs), N, generator=g)).half()
    Z = (7 + torch.rand(-(-K // gs), N, generator=g)).half()
    d = [t.to(dev) for t in (X, wn, P, S, Z)]
    stream = torch.cuda.current_stream(dev).cuda_stream
    best = int(L.mcq4_fused_rmsnorm_linear_int4_workspace_bytes(M, K, N, gs))
    least = 256 * 1024 + M * K * 2
    assert int(L.mcq4_matmul_int4_workspace_bytes(M, K, N, gs, _lib.MCQ4_DTYPE_F16)) == 0 and least < best

    def call(size):
        ws = torch.zeros(size + 512, dtype=torch.uint8, device=dev)
        base = -(-ws.data_ptr() // 256) * 256
        ws[base - ws.data_ptr() + size:] = 0x5A
        Y = torch.full((M, N), float("nan"), dtype=torch.float16, device=dev)
        st = L.mcq4_fused_rmsnorm_linear_int4(d[0].data_ptr(), K, d[1].data_ptr(), 1e-5, d[2].data_ptr(), d[3].data_ptr(), d[4].data_ptr(),
                                              _lib.MCQ4_DTYPE_F16, Y.data_ptr(), N, M, K, N, gs, base, size, stream)
        torch.cuda.synchronize(dev)
        assert bool((ws[base - ws.data_ptr() + size:] == 0x5A).all())
        return st, Y.double().cpu()

    assert call(least - 16)[0] == _lib.MCQ4_ERR_WORKSPACE
    (s0, y0), (s1, y1) = call(best), call(least)
    assert s0 == s1 == _lib.MCQ4_OK
    xn = (X.float() * torch.rsqrt((X.float() ** 2).mean(1, keepdim=True) + 1e-5) * wn.float()).double().abs()
    q = torch.stack([P & 15, P >> 4], 1).reshape(K, N).double()
    w = ((q - Z.double().repeat_interleave(gs, 0)[:K]) * S.double().repeat_interleave(gs, 0)[:K]).abs()
    assert bool(((y0 - y1).abs() <= 2.0 ** -10 * y0.abs() + 2 * K * 2.0 ** -24 * (xn @ w)).all())
