"""The conversion kernels (one or several columns per thread) against the oracles and, on
special values, against the rule in numpy (q4_0) and the one-column kernels, which an odd
row stride selects (INT4).

All exact: bytes, scales, zeros and outputs are compared bit for bit."""
import numpy as np
import pytest
import torch

from oracle import int4_ref as R
from oracle import q4_0_ref as Q

pytestmark = pytest.mark.gpu

TDT = {R.F32: torch.float32, R.F16: torch.float16, R.BF16: torch.bfloat16}


def _odd(w):
    """The same weight at a row stride that only the one-column kernels take."""
    s = torch.empty(w.shape[0], w.shape[1] + 1, dtype=w.dtype, device=w.device)
    s[:, :-1] = w
    return s[:, :-1]


def _bits(t):
    return t.contiguous().view(torch.uint8)


# Columns: one thread, the last column set of a workgroup, past it.  K: one block or group,
# a last group that is not whole.  From 384 K weights on INT4 dequantizes four columns a thread.
@pytest.mark.parametrize("K,N,gs", [(32, 4, 32), (64, 252, 64), (128, 260, 128), (160, 1028, 128), (288, 516, 64),
                                    (70, 8, 32), (4096, 1024, 128), (1030, 516, 32), (1550, 260, 128), (98310, 4, 64)])
@pytest.mark.parametrize("dtype", [R.F32, R.F16, R.BF16])
def test_wide_matches_oracle(dev, dtype, K, N, gs):
    import metalops_amd as mo
    print(f"convert {dtype} K={K} N={N} gs={gs}", flush=True)
    w = R.round_to(np.random.default_rng(K + N).standard_normal((K, N), np.float32) * 0.02, dtype)
    t = torch.from_numpy(w).to(TDT[dtype]).to(dev)
    p, s, z = mo.quantize_int4(t, gs)
    rp, rs, rz = R.quantize(w, gs, dtype)
    assert np.array_equal(p.cpu().numpy(), rp)
    assert np.array_equal(s.float().cpu().numpy(), rs) and np.array_equal(z.float().cpu().numpy(), rz)
    for out in (R.F32, R.F16, R.BF16):
        y = mo.dequantize_int4(p, s, z, gs, TDT[out])
        assert np.array_equal(y.float().cpu().numpy(), R.dequantize(rp, rs, rz, gs, out))
    if K % 32:
        return
    b = mo.quantize_ggml_q4_0(t)
    assert np.array_equal(b.cpu().numpy(), Q.quantize_ref_rule(w, {R.F32: "float32", R.F16: "float16", R.BF16: "bfloat16"}[dtype]))
    exact = Q.dequantize(b.cpu().numpy(), np.float32)
    for out in (R.F32, R.F16, R.BF16):
        y = mo.dequantize_ggml_q4_0(b, TDT[out])
        assert np.array_equal(y.float().cpu().numpy(), R.round_to(exact, out))


@pytest.mark.parametrize("dtype", [R.F32, R.F16, R.BF16])
@pytest.mark.parametrize("std", [0.02, 3e3, 1e-7])
def test_wide_matches_one_column_on_specials(dev, dtype, std):
    import metalops_amd as mo
    g = torch.Generator(device=dev).manual_seed(7)
    w = (torch.randn(512, 1024, generator=g, device=dev) * std * torch.exp(3 * torch.randn(1, 1024, generator=g, device=dev))).to(TDT[dtype])
    w[::97, ::31], w[::89, ::37], w[::83, ::41] = float("nan"), float("inf"), -float("inf")
    w[64:96], w[::53, ::3] = 0, -0.0
    assert torch.equal(mo.quantize_ggml_q4_0(w), mo.quantize_ggml_q4_0(_odd(w)))
    for gs in (32, 64, 128):
        for a, b in zip(mo.quantize_int4(w, gs), mo.quantize_int4(_odd(w), gs)):
            assert torch.equal(_bits(a), _bits(b))
    if dtype == R.F32:
        for a, b in zip(mo.quantize_to_int4(w, 128), mo.quantize_to_int4(_odd(w), 128)):
            assert torch.equal(_bits(a), _bits(b))


def _q4_rule(w, dtype):
    """The q4_0 rule of the kernels, a NaN weight left out of amax and coded 0: one IEEE operation and one
    rounding to the dtype per step."""
    x = w.reshape(w.shape[0] // 32, 32, w.shape[1])
    amax = np.fmax.reduce(np.abs(x), axis=1, initial=np.float32(0))
    d = R.round_to(amax / np.float32(7), dtype)
    d = np.where(d > 0, d, np.float32(1))
    t = R.round_to(R.round_to(x / d[:, None], dtype) + np.float32(8), dtype)
    q = np.fmin(np.fmax(np.rint(t), 0), 15).astype(np.uint8).reshape(x.shape[0], 8, 4, -1).astype(np.uint16)
    words = q[:, :, 0] | q[:, :, 1] << 4 | q[:, :, 2] << 8 | q[:, :, 3] << 12
    out = np.empty((x.shape[0], x.shape[2], 9), np.uint16)
    out[:, :, 0] = R.round_to(d, R.F16).astype(np.float16).view(np.uint16)
    out[:, :, 1:] = words.transpose(0, 2, 1)
    return out.view(np.uint8)


# Scales inside the range of the reciprocal form and outside it, and both in one wave.
@pytest.mark.parametrize("dtype", [R.F32, R.F16, R.BF16])
@pytest.mark.parametrize("std", [0.02, 3e3, 1e-7, 1e-25])
@pytest.mark.parametrize("N", [1, 257, 1024])
def test_q4_rule_on_specials(dev, dtype, std, N):
    import metalops_amd as mo
    g = torch.Generator().manual_seed(11)
    w = (torch.randn(320, N, generator=g) * std * torch.exp(6 * torch.randn(1, N, generator=g))).to(TDT[dtype])
    w[::97, ::31], w[::89, ::37], w[::83, ::41] = float("nan"), float("inf"), -float("inf")
    w[64:96], w[::53, ::3] = 0, -0.0
    with np.errstate(all="ignore"):
        want = _q4_rule(w.float().numpy(), dtype)
    assert np.array_equal(mo.quantize_ggml_q4_0(w.to(dev)).cpu().numpy(), want)


# Widths around two and four columns per thread, row strides and addresses that leave them, and the
# fp32 sizes (above 8 M and 11 M weights) on both sides of the idle-thread lines.
@pytest.mark.parametrize("K,N,pad,off", [(64, 2, 0, 0), (64, 510, 1, 0), (96, 514, 2, 1), (32, 1023, 0, 0), (64, 1026, 0, 2),
                                         (64, 260, 4, 0), (8224, 1024, 0, 0), (5504, 1536, 0, 0), (8224, 1024, 0, 1),
                                         (4704, 1792, 0, 0), (5664, 2056, 0, 0), (5664, 2044, 0, 0), (8480, 1364, 0, 0),
                                         (8480, 1368, 0, 0)])
def test_q4_dequantize_layouts(dev, K, N, pad, off):
    """dequantize through the C entry: padded rows and an `out` at an odd element."""
    from metalops_amd import _lib
    L = _lib.lib
    b = torch.randint(0, 256, (K // 32, N, 18), dtype=torch.uint8, generator=torch.Generator().manual_seed(K + N))
    b[:, :, 1] = (b[:, :, 1] & 0x83) | 0x20          # finite scales, both signs
    exact = Q.dequantize(b.numpy(), np.float32)
    d = b.to(dev)
    stream = torch.cuda.current_stream(dev).cuda_stream
    for out in (R.F32, R.F16, R.BF16):
        store = torch.full((K * (N + pad) + off + 8,), -1.0, dtype=TDT[out], device=dev)
        y = store[off:off + K * (N + pad)].view(K, N + pad)
        if out == R.BF16:
            st = L.mcq4_dequantize_q4_0_bf16(d.data_ptr(), K, N, y.data_ptr(), N + pad, stream)
        else:
            st = L.mcq4_dequantize_q4_0(d.data_ptr(), K, N, y.data_ptr(), N + pad,
                                        _lib.MCQ4_DTYPE_F16 if out == R.F16 else _lib.MCQ4_DTYPE_F32, stream)
        assert st == _lib.MCQ4_OK
        torch.cuda.synchronize(dev)
        want = R.round_to(exact, out)
        assert np.array_equal(y[:, :N].float().cpu().numpy(), want)
        assert np.array_equal(np.signbit(y[:, :N].float().cpu().numpy()), np.signbit(want))
        assert bool((store[:off] == -1).all()) and bool((y[:, N:] == -1).all()) and bool((store[-8:] == -1).all())
