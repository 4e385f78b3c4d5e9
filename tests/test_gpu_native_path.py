"""The native call path of the matmul functions (csrc/torch_ext/mcq4_torch.cpp) around
the kernels: its workspace, and what it leaves to the Python functions.
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
