"""INT4 / INT8 products between the decode kernels and the large tiles: bf16 prefill
(the bf16 instances of csrc/i4_gemm6.hip and i4_gemm7.hip) and fp16 up to 64 rows
(csrc/wx_skinny.hip).

Bar per output: W is the oracle's dequantized weight rounded once to X's dtype
(bit-exact in the kernels), so only fp32 sums and the output's rounding remain:
|Y - Y64| <= u |Y64| + K 2^-24 sum|x w|, u = 2^-8 (bf16), 2^-11 (fp16); a fused
activation (slope at most 1.13, fp32 evaluation) adds 2^-20 |y| and scales the second
term by 1.13.
"""
import numpy as np
import pytest
import torch

from oracle import int4_ref as R

pytestmark = pytest.mark.gpu

TDT = {R.F16: torch.float16, R.BF16: torch.bfloat16}
ULP = {R.F16: 2.0 ** -11, R.BF16: 2.0 ** -8}
ACT = {None: lambda y: y, "silu": lambda y: y / (1 + np.exp(-y)),
       "gelu": lambda y: 0.5 * y * (1 + np.tanh(np.sqrt(2 / np.pi) * (y + 0.044715 * y ** 3)))}


def _check(Y, X, W, xdt, act=None, E=0.0):
    X = X.double().numpy()
    W = np.asarray(W, np.float64)
    y = X @ W
    Yr, S = ACT[act](y), np.abs(X) @ np.abs(W)
    Y = Y.double().cpu().numpy()
    assert np.isfinite(Y).all()
    bound = ULP[xdt] * np.abs(Yr) + 1.13 * (X.shape[1] * 2.0 ** -24 * S + E) + (2.0 ** -20 * np.abs(y) if act else 0) + 1e-30
    bad = np.abs(Y - Yr) / bound
    assert bad.max() <= 1, f"err/bound {bad.max():.3g} at {np.unravel_index(bad.argmax(), bad.shape)}"


def _int4(dev, M, K, N, gs, xdt, sdt):
    w = R.round_to(np.random.default_rng(M * 3 + N).standard_normal((K, N), np.float32) * 0.02, sdt)
    p, s, z = R.quantize(w, gs, sdt)
    X = torch.randn(M, K, generator=torch.Generator().manual_seed(M + K)).to(TDT[xdt])
    args = [torch.from_numpy(p).to(dev)] + [torch.from_numpy(np.asarray(t, np.float32)).to(TDT[sdt]).to(dev) for t in (s, z)]
    return X, args, R.dequantize(p, s, z, gs, xdt)


# Rows around the line (64 / 65), the 128-row tile and the second tile; columns of one
# wave pair, of a workgroup with waves past N and of whole tiles; an odd number of K
# steps; eight, two and one K splits; the 256-row kernel by its switch.
@pytest.mark.parametrize("M,K,N,gs,sdt,env", [
    (65, 2048, 128, 128, R.BF16, {}), (127, 2080, 384, 32, R.BF16, {}), (129, 4096, 256, 128, R.F16, {}),
    (200, 2048, 16384, 128, R.BF16, {}), (200, 2048, 16384, 64, R.BF16, {"MCQ4_SPLIT_FOREIGN": "3"}),
    (300, 2080, 640, 160, R.BF16, {"MCQ4_I4_GEMM7": "1"}), (129, 4096, 256, 64, R.F16, {"MCQ4_I4_GEMM7": "1"}),
    (300, 2048, 5000, 128, R.BF16, {})])
def test_bf16_prefill(dev, monkeypatch, M, K, N, gs, sdt, env):
    import metalops_amd as mo
    from metalops_amd import _lib
    print(f"bf16 M={M} K={K} N={N} gs={gs} {env}", flush=True)
    for k in ("MCQ4_I4_GEMM6", "MCQ4_I4_GEMM7", "MCQ4_I4_PATH", "MCQ4_XCD_LOCAL"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    X, args, W = _int4(dev, M, K, N, gs, R.BF16, sdt)
    x = X.to(dev)
    Y = mo.matmul_int4(x, *args, gs)
    redone = _lib.split_fallback_count(reset=True)
    assert (redone > 0) == ("MCQ4_SPLIT_FOREIGN" in env)
    _check(Y, X, W, R.BF16)
    if not env:
        assert torch.equal(mo.matmul_int4(x, *args, gs).view(torch.int16), Y.view(torch.int16))


@pytest.mark.parametrize("M,K,N,gs,act", [(33, 96, 128, 32, None), (33, 4096, 384, 128, "silu"), (48, 2080, 256, 32, "gelu"),
                                          (64, 4096, 1024, 128, None), (33, 64, 16384, 32, None)])
def test_fp16_rows_int4(dev, M, K, N, gs, act):
    import metalops_amd as mo
    print(f"i4 f16 M={M} K={K} N={N} {act}", flush=True)
    X, args, W = _int4(dev, M, K, N, gs, R.F16, R.F16)
    f = {None: mo.matmul_int4, "silu": mo.matmul_int4_silu, "gelu": mo.matmul_int4_gelu}[act]
    _check(f(X.to(dev), *args, gs), X, W, R.F16, act)


@pytest.mark.parametrize("M,K,N,gs", [(17, 64, 128, 32), (32, 4096, 384, 128), (33, 2080, 256, 32), (64, 4096, 640, 128), (17, 512, 16512, 128)])
def test_fp16_rows_int8(dev, M, K, N, gs):
    import metalops_amd as mo
    print(f"i8 f16 M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(M + N)
    G = -(-K // gs)
    q = rng.integers(-128, 128, (K, N)).astype(np.int8)
    s = R.round_to(rng.uniform(0.5e-3, 2e-3, (G, N)).astype(np.float32), R.F16)
    z = R.round_to(rng.uniform(-20, 20, (G, N)).astype(np.float32), R.F16)
    X = torch.randn(M, K, generator=torch.Generator().manual_seed(M + K)).half()
    Y = mo.matmul_int8(X.to(dev), torch.from_numpy(q).to(dev), torch.from_numpy(s).half().to(dev), torch.from_numpy(z).half().to(dev), gs)
    _check(Y, X, R.dequantize_int8(q, s, z, gs, R.F16), R.F16)


# Beyond 16384 columns at short K, and above 56 rows with long K times wide N, the GEMM tiles
# take these rows: w = fma(q, s, c) with c = -z s rounded to fp16, so each weight is off W by at
# most 2^-11 (|z s| + 2 |W|) (c's rounding, the fma's, W's own).  Both sides of the column and K lines.
@pytest.mark.parametrize("wb,M,K,N,gs,act", [(4, 33, 64, 16512, 32, "silu"), (4, 48, 992, 16512, 32, None), (4, 48, 1024, 16512, 32, None),
                                             (4, 49, 1024, 16512, 128, None), (4, 64, 64, 24576, 32, "gelu"), (8, 17, 480, 16512, 32, None),
                                             (8, 33, 992, 16512, 32, None), (8, 40, 1024, 16512, 128, None), (8, 41, 1024, 16512, 128, None)])
def test_fp16_rows_gemm(dev, wb, M, K, N, gs, act):
    import metalops_amd as mo
    print(f"i{wb} f16 GEMM rows M={M} K={K} N={N} {act}", flush=True)
    rng = np.random.default_rng(M + N)
    G = -(-K // gs)
    s = rng.uniform(0.5e-3, 2e-3, (G, N)).astype(np.float16).astype(np.float32)
    z = rng.uniform(4, 12, (G, N)).astype(np.float16).astype(np.float32)
    X = torch.randn(M, K, generator=torch.Generator().manual_seed(M + K)).half()
    if wb == 4:
        p = rng.integers(0, 256, (K // 2, N), np.uint8)
        f, W = {None: mo.matmul_int4, "silu": mo.matmul_int4_silu, "gelu": mo.matmul_int4_gelu}[act], R.dequantize(p, s, z, gs, R.F16)
    else:
        p = rng.integers(-128, 128, (K, N)).astype(np.int8)
        f, W = mo.matmul_int8, R.dequantize_int8(p, s, z, gs, R.F16)
    Y = f(X.to(dev), torch.from_numpy(p).to(dev), torch.from_numpy(s).half().to(dev), torch.from_numpy(z).half().to(dev), gs)
    zs = np.repeat(np.abs(z * s), gs, axis=0)[:K]
    E = 2.0 ** -11 * (np.abs(X.float().numpy()) @ (zs + 2 * np.abs(np.asarray(W, np.float32)))).astype(np.float64)
    _check(Y, X, W, R.F16, act, E)
