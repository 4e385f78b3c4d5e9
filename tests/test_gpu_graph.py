"""HIP-graph capture and replay of the matmul entry points.

The kernels allocate nothing, record no memset, and leave their split-K
counters at zero, so a captured call must give the eager result on every
replay -- including replays with other (eager) work and synchronisations in
between, and split-K shapes whose counters are reused across replays.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mo(dev):
    import metalops_amd
    return metalops_amd


def _replay_check(dev, fn, out_ref, reps=4):
    s = torch.cuda.Stream(dev)
    with torch.cuda.stream(s):
        fn()                     # warm-up: per-stream workspace allocated before capture
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = fn()
    for r in range(reps):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.float().cpu().numpy(), out_ref, err_msg=f"replay {r}")
        # unrelated eager work between replays
        (torch.randn(1024, 1024, device=dev) @ torch.randn(1024, 1024, device=dev)).sum().item()


@pytest.mark.parametrize("M,K,N", [(1, 4096, 4096), (1, 4096, 128256 // 16), (8, 4096, 2048),
                                   (16, 14336, 4096), (128, 4096, 1024), (512, 11008, 512), (384, 4096, 4096),
                                   (512, 11008, 4096), (1024, 4096, 4096), (2048, 4096, 14336), (2048, 14336, 4096)])
def test_q4_0_graph_replay(mo, dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(M + N)
    W = torch.randn(K, N, generator=g, device=dev) * 0.02
    blocks = mo.quantize_ggml_q4_0_llama(W)
    X = torch.randn(M, K, generator=g, device=dev).half()
    ref = mo.matmul_ggml_q4_0(X, blocks).float().cpu().numpy()
    _replay_check(dev, lambda: mo.matmul_ggml_q4_0(X, blocks), ref)


@pytest.mark.parametrize("M,K,N", [(1, 4096, 4096), (16, 14336, 512), (1, 16384, 1024),
                                   (256, 4096, 1024), (128, 4096, 512)])
def test_int4_graph_replay(mo, dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(M + N)
    W = (torch.randn(K, N, generator=g, device=dev) * 0.02).half()
    gs = 32 if K == 16384 else 128          # K = 16384 with group 32 forces a decode K split
    packed, s, z = mo.quantize_int4(W, gs)
    X = torch.randn(M, K, generator=g, device=dev).half()
    ref = mo.matmul_int4(X, packed, s, z, gs).float().cpu().numpy()
    _replay_check(dev, lambda: mo.matmul_int4(X, packed, s, z, gs), ref)


def test_q4_0_grouped_graph_replay(mo, dev):
    """Gate and up in one launch, captured: every replay equals the eager call."""
    g = torch.Generator(device=dev).manual_seed(5)
    K, N = 4096, 11008
    blocks = [mo.quantize_ggml_q4_0_llama(torch.randn(K, N, generator=g, device=dev) * 0.02) for _ in range(2)]
    X = torch.randn(1, K, generator=g, device=dev).half()
    refs = [y.float().cpu().numpy() for y in mo.matmul_ggml_q4_0_grouped(X, blocks)]
    ref = np.concatenate(refs, axis=1)
    _replay_check(dev, lambda: torch.cat(mo.matmul_ggml_q4_0_grouped(X, blocks), dim=1), ref)


@pytest.mark.parametrize("M,K,N", [(1, 4096, 4096), (1, 11008, 4096), (4, 4096, 1024)])
def test_fused_rmsnorm_graph_replay(mo, dev, M, K, N):
    """The fused RMSNorm + INT4 linear (one launch at M = 1, two kernels above),
    captured: every replay equals the eager call."""
    g = torch.Generator(device=dev).manual_seed(M + K)
    W = (torch.randn(K, N, generator=g, device=dev) * 0.02).half()
    packed, s, z = mo.quantize_int4(W, 128)
    X = (torch.randn(M, K, generator=g, device=dev) * 2).half()
    wn = (1 + 0.1 * torch.randn(K, generator=g, device=dev)).half()
    ref = mo.fused_rmsnorm_linear_int4(X, wn, packed, s, z, 1e-5, 128).float().cpu().numpy()
    _replay_check(dev, lambda: mo.fused_rmsnorm_linear_int4(X, wn, packed, s, z, 1e-5, 128), ref)


# Calls whose K split uses a workspace that they can do without, and one that cannot.
def _graph_call(mo, dev, kind):
    from metalops_amd import _lib
    g = torch.Generator(device=dev).manual_seed(11)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    if kind[:2] == "q4":
        dt = {"q4_bf16": torch.bfloat16, "q4_f32": torch.float32, "q4_f16": torch.float16}[kind]
        M, K, N = (8, 14336, 4096) if dt == torch.bfloat16 else (33, 4096, 1024) if dt == torch.float32 else (17, 4096, 8192)
        X, W = rnd(M, K).to(dt), mo.quantize_ggml_q4_0_llama(rnd(K, N) * 0.02)
        code = {torch.bfloat16: _lib.MCQ4_DTYPE_BF16, torch.float32: _lib.MCQ4_DTYPE_F32, torch.float16: _lib.MCQ4_DTYPE_F16}[dt]
        return (lambda: mo.matmul_ggml_q4_0(X, W)), int(_lib.lib.mcq4_matmul_q4_0_workspace_bytes(M, K, N, code))
    M, K, N = 100, 4096, 1024
    X, w = rnd(M, K).bfloat16(), mo.quantize_int4((rnd(K, N) * 0.02).bfloat16(), 128)
    return (lambda: mo.matmul_int4(X, *w, 128)), int(_lib.lib.mcq4_matmul_int4_best_workspace_bytes(M, K, N, 128, _lib.MCQ4_DTYPE_BF16))


@pytest.mark.parametrize("kind", ["q4_bf16", "q4_f32", "q4_f16", "i4_bf16"])
@pytest.mark.parametrize("warm", [True, False])
def test_graph_keeps_its_workspace(mo, dev, kind, warm):
    """A captured call's workspace is the graph's own: a larger call on the stream, or a
    later capture there, frees nothing that a replay writes to."""
    from metalops_amd import _lib
    print(f"graph workspace {kind} warm={warm}", flush=True)
    fn, need = _graph_call(mo, dev, kind)
    Xb = torch.randn(512, 11008, device=dev).half()
    Wb = mo.quantize_ggml_q4_0_llama(torch.randn(11008, 512, device=dev) * 0.02)
    large = int(_lib.lib.mcq4_matmul_workspace_bytes(512, 11008, 512))
    assert 0 < need < large and large > 1 << 20
    ref, big_ref = fn(), mo.matmul_ggml_q4_0(Xb, Wb)
    torch.cuda.synchronize()
    s = torch.cuda.Stream(dev)
    if warm:
        with torch.cuda.stream(s):
            fn()
    torch.cuda.synchronize()
    graphs, outs = [], []
    for _ in range(2):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1], stream=s):
            outs.append(fn())
    with torch.cuda.stream(s):
        first = fn()                         # before any replay: the counters are zero
        big = mo.matmul_ggml_q4_0(Xb, Wb)    # replaces the stream's buffer
        fresh = [torch.full((1 << 20,), 0x5A, dtype=torch.uint8, device=dev) for _ in range(8 + 2 * large // (1 << 20))]
    torch.cuda.synchronize()
    assert torch.equal(first, ref) and torch.equal(big, big_ref)
    for _ in range(3):
        for g, out in zip(graphs, outs):
            out.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref)
    assert all(bool((t == 0x5A).all()) for t in fresh)


# Splits that a second launch sums: those that one kernel exchanges may be recomputed
# beside other work, in another order of the sums.
@pytest.mark.parametrize("kind", ["q4_f32", "i4_bf16"])
def test_replay_beside_eager_calls(mo, dev, kind):
    """Replays on another stream than the capture's, eager calls on the capture's: each has its own workspace."""
    print(f"replay beside eager {kind}", flush=True)
    fn, _ = _graph_call(mo, dev, kind)
    ref = fn()
    s, r = torch.cuda.Stream(dev), torch.cuda.Stream(dev)
    with torch.cuda.stream(s):
        fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = fn()
    for _ in range(20):
        with torch.cuda.stream(r):
            g.replay()
        with torch.cuda.stream(s):
            ys = [fn() for _ in range(3)]
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and all(torch.equal(y, ref) for y in ys)
