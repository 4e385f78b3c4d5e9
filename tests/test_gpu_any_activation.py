"""The kernels for every activation dtype, column count and alignment (csrc/wx_*.hip)
against the CPU oracles: bf16 and fp32 activations, fp16 ones at column counts the
fp16 kernels leave.

Bar per output: W is the oracle's dequantized weight rounded once to X's dtype
(bit-exact in the kernels), so only fp32 sums and the output's rounding remain:
|Y - Y64| <= u |Y64| + K 2^-24 sum|x w|, u = 2^-8 (bf16), 2^-11 (fp16), 2^-23 (fp32).
"""
import numpy as np
import pytest
import torch

from oracle import int4_ref as R
from oracle import q4_0_ref as Q

pytestmark = pytest.mark.gpu

TDT = {R.F32: torch.float32, R.F16: torch.float16, R.BF16: torch.bfloat16}
ULP = {R.F32: 2.0 ** -23, R.F16: 2.0 ** -11, R.BF16: 2.0 ** -8}


def _x(M, K, xdt, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, K, generator=g).to(TDT[xdt])


def _check(Y, X, W, xdt, act=None):
    X = X.double().numpy()
    W = np.asarray(W, np.float64)
    Yr, S = X @ W, np.abs(X) @ np.abs(W)
    Y = Y.double().cpu().numpy()
    assert np.isfinite(Y).all()
    bound = ULP[xdt] * np.abs(Yr) + X.shape[1] * 2.0 ** -24 * S + 1e-30
    bad = np.abs(Y - Yr) / bound
    assert bad.max() <= 1, f"err/bound {bad.max():.3g} at {np.unravel_index(bad.argmax(), bad.shape)}"


# Rows: the smallest, around 32 and 64 (row tiles, the decode / prefill line), around
# 128 (row tile of the prefill kernel).  Columns: 1, around 64 and 256 (column tiles),
# odd.  K: one block, an odd number of blocks, splits over workgroups.
# Spans of 0..4 column groups (N = 48, 4096, 8208, 16384 at K <= 4096) and their K split
# (N <= 4096, long K).
SHAPES = [(1, 4096, 48), (4, 2080, 4096), (9, 1024, 8208), (8, 288, 16384), (1, 8224, 4096), (13, 14336, 1024), (1, 32, 1), (1, 4096, 257), (3, 96, 63), (16, 2080, 64), (31, 1024, 65), (32, 4096, 128), (33, 64, 130),
          (64, 4128, 100), (65, 32, 255), (65, 1056, 257), (127, 992, 256), (129, 2080, 513), (300, 4096, 40)]


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("xdt", [R.BF16, R.F32, R.F16])
def test_q4(dev, xdt, M, K, N):
    import metalops_amd as mo
    print(f"q4 {xdt} M={M} K={K} N={N}", flush=True)
    w = np.random.default_rng(M * 7 + N).standard_normal((K, N), np.float32) * 0.02
    b = Q.quantize_llama_rule(w)
    X = _x(M, K, xdt, M + K)
    Y = mo.matmul_ggml_q4_0(X.to(dev), torch.from_numpy(b).to(dev))
    if xdt == R.F16 and M <= 32:       # decode kernels: unrounded weights, d applied to the sums
        W = Q.dequantize(b, np.float32)
        Yr = X.double().numpy() @ W.astype(np.float64)
        assert (np.abs(Y.double().cpu().numpy() - Yr) <= 1e-2 * np.abs(Yr).max(1, keepdims=True)).all()
        return
    _check(Y, X, R.round_to(Q.dequantize(b, np.float32), xdt), xdt)


# Fewer columns than one wave's 64 (N % 8 == 0): the prefill tiles' other waves have none; a
# K split, one K step, two row tiles.
@pytest.mark.parametrize("M,K,N", [(65, 4096, 8), (65, 32, 24), (130, 1056, 56), (300, 4096, 72)])
@pytest.mark.parametrize("xdt", [R.BF16, R.F16])
def test_q4_narrow_prefill(dev, xdt, M, K, N):
    import metalops_amd as mo
    print(f"q4 narrow {xdt} M={M} K={K} N={N}", flush=True)
    w = np.random.default_rng(M + N).standard_normal((K, N), np.float32) * 0.02
    b = Q.quantize_llama_rule(w)
    X = _x(M, K, xdt, M + K)
    Y = mo.matmul_ggml_q4_0(X.to(dev), torch.from_numpy(b).to(dev))
    _check(Y, X, R.round_to(Q.dequantize(b, np.float32), xdt), xdt)


# fp16, 17..32 rows, whole 16-byte weight rows: the weight stays unrounded (exact block
# sums, d applied in fp32), so the bar is that of fp32 sums against (q - 8) d itself.
# Then 33..64 rows on both sides of each line of the dispatch: strips (unrounded too), the
# kernel above them, prefill tiles beyond 16384 columns; the few-tile kernel's round.
# Then weights the strip kernels do not take, on both sides of the K from which wx runs them.
@pytest.mark.parametrize("M,K,N,exact", [(17, 4096, 8, True), (24, 4096, 136, True), (32, 14336, 64, True), (31, 4128, 4096, True),
                                         (33, 2528, 16, True), (64, 1024, 4096, True), (48, 32, 8, False), (33, 2560, 16, False),
                                         (40, 1024, 4112, False), (64, 2048, 24, False), (33, 224, 16392, False),
                                         (64, 256, 16392, False), (57, 256, 24576, False), (56, 256, 24576, False), (64, 2016, 32, True), (64, 2048, 32, False),
                                         (1, 4096, 33, False), (16, 4128, 257, False), (17, 4096, 65, False), (64, 4096, 1025, False),
                                         (4, 4096, 33, False), (5, 4096, 33, False), (5, 5120, 33, False), (9, 10208, 33, False),
                                         (9, 10240, 33, False), (16, 4096, 4097, False), (40, 5120, 65, False), (41, 4096, 65, False)])
def test_q4_fp16_rows(dev, M, K, N, exact):
    import metalops_amd as mo
    print(f"q4 fp16 M={M} K={K} N={N}", flush=True)
    w = np.random.default_rng(M * 5 + N).standard_normal((K, N), np.float32) * 0.02
    b = Q.quantize_llama_rule(w)
    X = _x(M, K, R.F16, M + K)
    Y = mo.matmul_ggml_q4_0(X.to(dev), torch.from_numpy(b).to(dev))
    W = Q.dequantize(b, np.float32)
    _check(Y, X, W if exact else R.round_to(W, R.F16), R.F16)


# Prefill on both sides of the short-K lines: N % 8 == 0 (K = 160, 128 tiles of 128 x 256), odd (K = 384,
# up to 144 tiles, 160 up to 288), and the K split of 1 M outputs (K = 768).
@pytest.mark.parametrize("M,K,N", [(65, 32, 8), (130, 128, 136), (130, 160, 136), (2048, 96, 2048 + 8), (65, 32, 1), (129, 352, 257),
                                   (129, 384, 257), (1100, 352, 4001), (1153, 128, 4001), (1153, 160, 4001), (4736, 96, 2047), (1100, 736, 1001),
                                   (1100, 768, 1001)])
@pytest.mark.parametrize("xdt", [R.F16, R.BF16])
def test_q4_short_k(dev, xdt, M, K, N):
    import metalops_amd as mo
    print(f"q4 short K {xdt} M={M} K={K} N={N}", flush=True)
    w = np.random.default_rng(M + N).standard_normal((K, N), np.float32) * 0.02
    b = Q.quantize_llama_rule(w)
    X = _x(M, K, xdt, M + K)
    Y = mo.matmul_ggml_q4_0(X.to(dev), torch.from_numpy(b).to(dev))
    _check(Y, X, R.round_to(Q.dequantize(b, np.float32), xdt), xdt)


@pytest.mark.parametrize("M,K,N,pad,off", [(5, 256, 33, 3, 0), (40, 256, 66, 8, 1), (100, 544, 70, 5, 3), (70, 512, 64, 0, 2)])
@pytest.mark.parametrize("xdt", [R.BF16, R.F32])
def test_q4_row_strides(dev, xdt, M, K, N, pad, off):
    """Activations at a row stride and offset that are no multiple of 16 bytes; odd weight address."""
    import metalops_amd as mo
    print(f"q4 strides {xdt} M={M} K={K} N={N} pad={pad} off={off}", flush=True)
    w = np.random.default_rng(M).standard_normal((K, N), np.float32) * 0.02
    b = Q.quantize_ref_rule(w)
    store = torch.zeros(M * (K + pad) + off, dtype=TDT[xdt])
    X = _x(M, K, xdt, M)
    view = store[off:].view(M, K + pad)[:, :K]
    view.copy_(X)
    d = store.to(dev)[off:].view(M, K + pad)[:, :K]
    raw = torch.zeros(b.size + 2, dtype=torch.uint8)
    raw[2:] = torch.from_numpy(b.reshape(-1))
    blocks = raw.to(dev)[2:].view(b.shape)
    _check(mo.matmul_ggml_q4_0(d, blocks), X, R.round_to(Q.dequantize(b, np.float32), xdt), xdt)


GSHAPES = [(1, 64, 2), (2, 96, 63), (17, 2048, 130), (32, 4100, 128), (33, 1024, 65), (64, 4096, 66), (65, 64, 3),
           (66, 544, 257), (129, 1030, 514), (260, 4096, 130)]


@pytest.mark.parametrize("M,K,N", GSHAPES)
@pytest.mark.parametrize("xdt,sdt,gs", [(R.BF16, R.BF16, 128), (R.F32, R.F32, 64), (R.F16, R.F16, 32), (R.BF16, R.F32, 32),
                                        (R.F32, R.F16, 256)])
def test_int4(dev, xdt, sdt, gs, M, K, N):
    import metalops_amd as mo
    print(f"i4 {xdt}/{sdt} gs={gs} M={M} K={K} N={N}", flush=True)
    w = R.round_to(np.random.default_rng(M * 3 + N).standard_normal((K, N), np.float32) * 0.02, sdt)
    p, s, z = R.quantize(w, gs, sdt)
    X = _x(M, K, xdt, M + K)
    args = [torch.from_numpy(p).to(dev)] + [torch.from_numpy(np.asarray(t, np.float32)).to(TDT[sdt]).to(dev) for t in (s, z)]
    Y = mo.matmul_int4(X.to(dev), *args, gs)
    if xdt == R.F16 and K % 32 == 0 and (N % 128 == 0 or M <= 16 and N % 8 == 0):
        return                         # the fp16 kernels' own tests
    _check(Y, X, R.dequantize(p, s, z, gs, xdt), xdt)


@pytest.mark.parametrize("M,K,N", [(1, 33, 2), (9, 515, 67), (40, 2048, 130), (130, 1031, 259), (200, 640, 64)])
@pytest.mark.parametrize("xdt,sdt,gs", [(R.BF16, R.BF16, 128), (R.F32, R.F32, 32), (R.F16, R.F32, 64)])
def test_int8(dev, xdt, sdt, gs, M, K, N):
    import metalops_amd as mo
    print(f"i8 {xdt}/{sdt} gs={gs} M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(M + N)
    G = -(-K // gs)
    q = rng.integers(-128, 128, (K, N)).astype(np.int8)
    s = R.round_to(rng.uniform(0.5e-3, 2e-3, (G, N)).astype(np.float32), sdt)
    z = R.round_to(rng.uniform(-20, 20, (G, N)).astype(np.float32), sdt)
    X = _x(M, K, xdt, M + K)
    Y = mo.matmul_int8(X.to(dev), torch.from_numpy(q).to(dev), torch.from_numpy(s).to(TDT[sdt]).to(dev),
                       torch.from_numpy(z).to(TDT[sdt]).to(dev), gs)
    if xdt == R.F16 and K % 32 == 0 and (N % 128 == 0 or M <= 16 and N % 8 == 0):
        return
    _check(Y, X, R.dequantize_int8(q, s, z, gs, xdt), xdt)


# wx_gemv / wx_gemm at an odd width; then, in bf16, the kernels of aligned widths: spans (whole and
# split K), wx_mid (both row forms), q4_gemm6, q4_gemm7 (its ragged form) and q4_gemm8.
@pytest.mark.parametrize("M,K,N,env", [(4, 96, 70, {}), (100, 96, 70, {}), (1, 96, 48, {}), (4, 96, 64, {}), (16, 96, 64, {}),
                                       (9, 8224, 64, {}), (24, 96, 72, {}), (40, 96, 64, {}), (100, 96, 72, {}),
                                       (100, 96, 128, {"MCQ4_GEMM_PATH": "7"}), (100, 96, 72, {"MCQ4_GEMM_PATH": "7"}),
                                       (100, 96, 128, {"MCQ4_GEMM_PATH": "8"})])
@pytest.mark.parametrize("xdt", [R.BF16, R.F32])
def test_non_finite(dev, monkeypatch, xdt, M, K, N, env):
    """Infinities and NaN stay in their own rows and columns: an inf activation, a block scale of inf."""
    import metalops_amd as mo
    print(f"non-finite {xdt} M={M} K={K} N={N} {env}", flush=True)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    w = np.random.default_rng(5).standard_normal((K, N), np.float32) * 0.02
    b = Q.quantize_ref_rule(w)
    b[1, 7, :2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    b[1, 7, 2:] = 0xFF                 # q = 15 everywhere: +inf weights
    X = _x(M, K, xdt, 9).abs() + 0.1
    if M > 2:
        X[1, 40] = float("inf")
        X[2, 3] = float("nan")
    Y = mo.matmul_ggml_q4_0(X.to(dev), torch.from_numpy(b).to(dev)).double().cpu().numpy()
    with np.errstate(all="ignore"):
        W = R.round_to(Q.dequantize(b, np.float32), xdt).astype(np.float64)
        Yr = np.stack([(X[m].double().numpy()[:, None] * W).sum(0) for m in range(M)])
    assert np.array_equal(np.isnan(Y), np.isnan(Yr))
    inf = np.isinf(Yr)
    assert inf.any() and np.array_equal(Y[inf], Yr[inf]) and np.isfinite(Y[~inf & ~np.isnan(Yr)]).all()
