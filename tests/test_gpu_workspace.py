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
