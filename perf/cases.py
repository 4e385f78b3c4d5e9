"""Performance cases: the calls that a program using metalops_amd makes, over their real range.

The listed cases are the work of serving a quantized model, each through the
package's public functions: single-row decode (where latency and launches
count), small-batch decode, prefill, weight conversion at load time, and the
per-group INT4 layer.  Shapes are those of ``bench.py`` and of the tests.
``draw`` gives further cases of the same ranges: every operation, activation
dtype, scale dtype and group size, sizes spread over their logarithm, column
counts that are multiples of 128, multiples of 8 and odd.

Weights are quantized here in plain torch (the formats' own rules), so the
64-bit results of ``exact`` use none of the package's code.
"""
import math

import torch

import metalops_amd as mo

_DT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
_DEV = "cuda"
# The largest listed product (M = 2048, 4096 x 14336); no drawn case does more.
_MOST_FLOPS = 2 * 2048 * 4096 * 14336
# bf16 and fp32 activations, fp32 scales and INT8 weights serve smaller jobs.
_MOST_FLOPS_OTHER = _MOST_FLOPS // 8

# The five projections of a Llama-2-7B layer: (K, N).
_LAYER = {"qkv": (4096, 12288), "o": (4096, 4096), "gate": (4096, 11008), "up": (4096, 11008),
          "down": (11008, 4096)}


def listed():
    return [
        # The smallest call: one attention output projection of a decode step.
        {"name": "q4_o_m1", "op": "q4", "x": "f16", "M": 1, "K": 4096, "N": 4096},
        # A decode step's projections of one layer, gate and up in one call: the headline workload.
        {"name": "q4_layer_m1", "op": "q4_layer", "x": "f16", "M": 1},
        # Batched decode, long K: the down projection for 16 sequences.
        {"name": "q4_down_m16", "op": "q4", "x": "f16", "M": 16, "K": 14336, "N": 4096},
        # A larger decode batch (or draft verification): between the decode and the prefill sizes.
        {"name": "q4_up_m48", "op": "q4", "x": "f16", "M": 48, "K": 4096, "N": 14336},
        # Prefill of a long prompt: the largest call.
        {"name": "q4_up_m2048", "op": "q4", "x": "f16", "M": 2048, "K": 4096, "N": 14336},
        # A prompt and a width that are whole tiles of nothing: N is a multiple of 8 only.
        {"name": "q4_ragged_m300", "op": "q4", "x": "f16", "M": 300, "K": 11008, "N": 4104},
        # A bf16 model decoding for a few sequences.
        {"name": "q4_bf16_m4", "op": "q4", "x": "bf16", "M": 4, "K": 4096, "N": 11008},
        # A bf16 model's prefill.
        {"name": "q4_bf16_m512", "op": "q4", "x": "bf16", "M": 512, "K": 4096, "N": 4096},
        # Loading a model: a bf16 weight quantized, and blocks expanded for a dense layer.
        {"name": "q4_load", "op": "q4_load", "w": "bf16", "out": "f16", "K": 4096, "N": 14336},
        # A decode step's projections of one layer with per-group INT4 weights and the fused calls.
        {"name": "i4_layer_m1", "op": "i4_layer", "x": "f16", "s": "f16", "gs": 128, "M": 1},
        # Int4Linear of a bf16 module on a batch of short prompts, weights kept quantized.
        {"name": "i4_linear_bf16", "op": "i4_linear", "x": "bf16", "s": "bf16", "gs": 128, "B": 4,
         "M": 64, "K": 4096, "N": 11008},
        # Int4Linear of a module in torch's default dtype (fp32 activations and scales).
        {"name": "i4_linear_f32", "op": "i4_linear", "x": "f32", "s": "f32", "gs": 128, "B": 1,
         "M": 32, "K": 4096, "N": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["q4", "q4", "q4", "q4", "i4", "i4", "i4_linear", "i4_norm", "i8", "q4_load", "i4_load",
                     "q4_group"])
    K = 128 * _log(rng, 8, 112) if rng.random() < 0.6 else 32 * _log(rng, 32, 448)
    if op[:2] != "q4" and rng.random() < 0.15:
        K += 2 * rng.randrange(1, 16)            # a last group that is not whole
    if op == "i8" and K % 2 == 0 and rng.random() < 0.1:
        K += 1
    r = rng.random()
    N = 128 * _log(rng, 8, 112) if r < 0.6 else 8 * _log(rng, 128, 1792) if r < 0.85 else _log(rng, 1024, 14336)
    M = _log(rng, 1, 2048)
    x = rng.choice(["f16", "f16", "f16", "bf16", "bf16", "f32"])
    gs = rng.choice([32, 64, 128, 128])
    if op == "q4":
        case = {"op": op, "x": x, "M": M, "K": K, "N": N}
    elif op == "q4_group":
        return {"op": op, "x": x, "M": _log(rng, 1, 8), "K": K, "N": N, "count": rng.randrange(2, 5)}
    elif op in ("q4_load", "i4_load"):
        K = min(K, 4096 * 14336 // N // 128 * 128)   # no larger weight than the listed one
        w, out = rng.choice(["f32", "f16", "bf16"]), rng.choice(["f16", "f32", "bf16"])
        return {"op": op, "w": w, "out": out, **({"gs": gs} if op == "i4_load" else {}), "K": K, "N": N}
    elif op == "i4_linear":
        case = {"op": op, "x": x, "s": x, "gs": gs, "B": rng.choice([1, 2, 3]), "M": max(1, M // 4), "K": K, "N": N}
    elif op == "i4_norm":
        case = {"op": op, "x": "f16", "s": rng.choice(["f16", "f32"]), "gs": gs, "M": _log(rng, 1, 64), "K": K,
                "N": N}
    elif op == "i4":
        act = rng.choice(["none", "none", "silu", "gelu"]) if x == "f16" else "none"
        case = {"op": op, "x": x, "s": rng.choice([x, x, "f32"]), "gs": gs, "act": act, "M": M, "K": K, "N": N}
    else:
        case = {"op": op, "x": x, "s": rng.choice([x, x, "f32"]), "gs": gs, "M": M, "K": K, "N": N}
    main = x == "f16" and case.get("s", x) == x and op != "i8" and N % 128 == 0
    most = _MOST_FLOPS if main else _MOST_FLOPS_OTHER
    rows = case["M"] * case.get("B", 1)
    if 2 * rows * K * N > most:
        case["M"] = max(1, int(case["M"] * most / (2 * rows * K * N)))
    return case


# ---- inputs ------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=_DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(*shape, generator=g, device=_DEV) * std).to(dtype)


def _q4_blocks(w):
    """[K, N] fp32 -> [K/32, N, 18] uint8 blocks (scale = amax/7, nibbles in element order)."""
    K, N = w.shape
    b = w.reshape(K // 32, 32, N)
    d = b.abs().amax(1) / 7
    d = torch.where(d > 0, d, torch.ones_like(d))
    q = (b / d[:, None] + 8).round().clamp(0, 15).to(torch.uint8)
    out = torch.empty(K // 32, N, 18, dtype=torch.uint8, device=w.device)
    out[..., :2] = d.half().view(torch.uint8).reshape(K // 32, N, 2)
    out[..., 2:] = (q[:, 0::2] | (q[:, 1::2] << 4)).permute(0, 2, 1)
    return out


def _q4_values(blocks):
    """The exact (q - 8)*d of every weight, fp64 [K, N]."""
    nb, N, _ = blocks.shape
    d = blocks[..., :2].contiguous().view(torch.float16).reshape(nb, 1, N).double()
    by = blocks[..., 2:].permute(0, 2, 1)
    q = torch.stack([by & 15, by >> 4], 2).reshape(nb, 32, N).double()
    return ((q - 8) * d).reshape(nb * 32, N)


def _grouped(w, gs, levels):
    """Per group and column: whole-number codes, scales and zeros of [K, N] fp32."""
    K, N = w.shape
    G = -(-K // gs)
    pad = G * gs - K
    wp = torch.cat([w, w[-1:].expand(pad, N)]) if pad else w
    wg = wp.reshape(G, gs, N)
    mn, mx = wg.amin(1), wg.amax(1)
    s = ((mx - mn) / levels).clamp(min=1e-8)
    return wg, mn, s, K


def _int4(w, gs, dtype):
    wg, mn, s, K = _grouped(w, gs, 15)
    z = -mn / s
    q = (wg / s[:, None] + z[:, None]).round().clamp(0, 15).to(torch.uint8).reshape(-1, w.shape[1])[:K]
    return q[0::2] | (q[1::2] << 4), s.to(dtype), z.to(dtype)


def _int8(w, gs, dtype):
    wg, mn, s, K = _grouped(w, gs, 255)
    z = -mn / s - 128
    q = (wg / s[:, None] + z[:, None]).round().clamp(-128, 127).to(torch.int8).reshape(-1, w.shape[1])[:K]
    return q, s.to(dtype), z.to(dtype)


def _group_values(q, scales, zeros, gs):
    """The exact (q - zero)*scale of every weight, fp64 [K, N]."""
    g = torch.arange(q.shape[0], device=q.device) // gs
    return (q.double() - zeros.double()[g]) * scales.double()[g]


def _nibbles(packed):
    return torch.stack([packed & 15, packed >> 4], 1).reshape(-1, packed.shape[1])


def prepare(case, seed):
    g, op = _gen(seed), case["op"]
    st = {"case": case}
    if op in ("q4", "q4_group"):
        st["x"] = _randn(g, case["M"], case["K"], dtype=_DT[case["x"]])
        n = case.get("count", 1)
        st["w"] = [_q4_blocks(_randn(g, case["K"], case["N"], std=0.02)) for _ in range(n)]
    elif op == "q4_layer":
        for k, (K, N) in _LAYER.items():
            st[k] = _q4_blocks(_randn(g, K, N, std=0.02))
        for k, n in (("x", 4096), ("a", 4096), ("h", 4096), ("f", 11008)):
            st[k] = _randn(g, case["M"], n, dtype=torch.float16)
    elif op == "q4_load":
        st["weight"] = _randn(g, case["K"], case["N"], dtype=_DT[case["w"]], std=0.02)
        st["blocks"] = _q4_blocks(_randn(g, case["K"], case["N"], std=0.02))
    elif op == "i4_load":
        st["weight"] = _randn(g, case["K"], case["N"], dtype=_DT[case["w"]], std=0.02)
        st["packed"] = _int4(_randn(g, case["K"], case["N"], std=0.02), case["gs"], _DT[case["w"]])
    elif op == "i4_layer":
        for k, (K, N) in _LAYER.items():
            st[k] = _int4(_randn(g, K, N, std=0.02), case["gs"], _DT[case["s"]])
        for k, n in (("x", 4096), ("a", 4096), ("h", 4096), ("f", 11008)):
            st[k] = _randn(g, case["M"], n, dtype=torch.float16)
        st["norm"] = (1 + _randn(g, 4096, std=0.1)).half()
    elif op == "i4_linear":
        layer = mo.Int4Linear(case["K"], case["N"], group_size=case["gs"], bias=True, device=_DEV, dtype=_DT[case["s"]])
        packed, s, z = _int4(_randn(g, case["K"], case["N"], std=0.02), case["gs"], _DT[case["s"]])
        for name, t in (("weight_packed", packed), ("scales", s), ("zeros", z),
                        ("bias", _randn(g, case["N"], std=0.1))):
            getattr(layer, name).copy_(t)
        layer.keep_quantized()
        st["layer"] = layer
        st["x"] = _randn(g, case["B"], case["M"], case["K"], dtype=_DT[case["x"]])
    else:
        make = _int8 if op == "i8" else _int4
        st["w"] = make(_randn(g, case["K"], case["N"], std=0.02), case["gs"], _DT[case["s"]])
        st["x"] = _randn(g, case["M"], case["K"], dtype=_DT[case["x"]])
        if op == "i4_norm":
            st["norm"] = (1 + _randn(g, case["K"], std=0.1)).half()
    return st


# ---- one pass ----------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    op = case["op"]
    if op == "q4":
        return mo.matmul_ggml_q4_0(state["x"], state["w"][0])
    if op == "q4_group":
        return mo.matmul_ggml_q4_0_grouped(state["x"], state["w"])
    if op == "q4_layer":
        return {"qkv": mo.matmul_ggml_q4_0(state["x"], state["qkv"]),
                "o": mo.matmul_ggml_q4_0(state["a"], state["o"]),
                "gate_up": mo.matmul_ggml_q4_0_grouped(state["h"], [state["gate"], state["up"]]),
                "down": mo.matmul_ggml_q4_0(state["f"], state["down"])}
    if op == "q4_load":
        return [mo.quantize_ggml_q4_0(state["weight"]),
                mo.dequantize_ggml_q4_0(state["blocks"], _DT[case["out"]])]
    if op == "i4_load":
        p, s, z = state["packed"]
        return [*mo.quantize_int4(state["weight"], case["gs"]),
                mo.dequantize_int4(p, s, z, case["gs"], _DT[case["out"]])]
    if op == "i4_layer":
        gs = case["gs"]
        return {"qkv": mo.fused_rmsnorm_linear_int4(state["x"], state["norm"], *state["qkv"], 1e-5, gs),
                "o": mo.matmul_int4(state["a"], *state["o"], gs),
                "gate": mo.matmul_int4_silu(state["h"], *state["gate"], gs),
                "up": mo.matmul_int4(state["h"], *state["up"], gs),
                "down": mo.matmul_int4(state["f"], *state["down"], gs)}
    if op == "i4_linear":
        return state["layer"](state["x"])
    if op == "i4_norm":
        return mo.fused_rmsnorm_linear_int4(state["x"], state["norm"], *state["w"], 1e-5, case["gs"])
    if op == "i8":
        return mo.matmul_int8(state["x"], *state["w"], case["gs"])
    fn = {"none": mo.matmul_int4, "silu": mo.matmul_int4_silu, "gelu": mo.matmul_int4_gelu}[case["act"]]
    return fn(state["x"], *state["w"], case["gs"])


# ---- what a pass cannot do without ---------------------------------------------------------------

_ES = {"f16": 2, "bf16": 2, "f32": 4}


def _weight_bytes(case, K, N):
    if case["op"][:2] == "q4":
        return 18 * (K // 32) * N
    groups = -(-K // case["gs"])
    return (K * N if case["op"] == "i8" else K // 2 * N) + 2 * groups * N * _ES[case["s"]]


def work(case):
    op = case["op"]
    if op in ("q4_load", "i4_load"):
        K, N = case["K"], case["N"]
        if op == "q4_load":
            packed = 18 * (K // 32) * N
        else:
            packed = K // 2 * N + 2 * -(-K // case["gs"]) * N * _ES[case["w"]]
        return {"bytes": K * N * (_ES[case["w"]] + _ES[case["out"]]) + 2 * packed, "flops": 0}
    if op in ("q4_layer", "i4_layer"):
        M = case["M"]
        byt = sum(_weight_bytes(case, K, N) + 2 * M * N for K, N in _LAYER.values()) + 2 * M * (3 * 4096 + 11008)
        return {"bytes": byt, "flops": sum(2 * M * K * N for K, N in _LAYER.values())}
    M, K, N, es = case["M"] * case.get("B", 1), case["K"], case["N"], _ES[case["x"]]
    n = case.get("count", 1)
    return {"bytes": n * _weight_bytes(case, K, N) + es * M * (K + n * N), "flops": 2 * n * M * K * N}


def tolerance(case):
    if case["op"] in ("q4_load", "i4_load"):
        return "exact"
    # Another summation order and weights rounded to the activations' dtype or not.
    return {"f16": {"rel": 2e-3, "max": 0.02}, "bf16": {"rel": 1e-2, "max": 0.1},
            "f32": {"rel": 4e-6, "max": 4e-5}}[case["x"]]


def _act(y, act):
    if act == "silu":
        return y / (1 + torch.exp(-y))
    if act == "gelu":
        return 0.5 * y * (1 + torch.tanh(math.sqrt(2 / math.pi) * (y + 0.044715 * y ** 3)))
    return y


def exact(case, seed):
    """The 64-bit results: weights rounded to the activations' dtype, as the formats' dense form has them."""
    op = case["op"]
    if op in ("q4_load", "i4_load"):
        return None
    st = prepare(case, seed)
    dt = _DT[case["x"]]

    def dense(values):
        return values.to(dt).double()

    def i4(x, w, act="none"):
        p, s, z = w
        q = p if op == "i8" else _nibbles(p)
        return _act(x.double() @ dense(_group_values(q, s, z, case["gs"])), act)

    def norm(x):
        x = x.double()
        return (x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * st["norm"].double()).half()

    if op == "q4":
        return st["x"].double() @ dense(_q4_values(st["w"][0]))
    if op == "q4_group":
        return [st["x"].double() @ dense(_q4_values(w)) for w in st["w"]]
    if op == "q4_layer":
        def q4(x, w):
            return st[x].double() @ dense(_q4_values(st[w]))
        return {"qkv": q4("x", "qkv"), "o": q4("a", "o"), "gate_up": [q4("h", "gate"), q4("h", "up")],
                "down": q4("f", "down")}
    if op == "i4_layer":
        return {"qkv": i4(norm(st["x"]), st["qkv"]), "o": i4(st["a"], st["o"]), "gate": i4(st["h"], st["gate"], "silu"),
                "up": i4(st["h"], st["up"]), "down": i4(st["f"], st["down"])}
    if op == "i4_linear":
        y = st["layer"]
        return i4(st["x"], (y.weight_packed, y.scales, y.zeros)) + y.bias.double()
    if op == "i4_norm":
        return i4(norm(st["x"]), st["w"])
    return i4(st["x"], st["w"], case.get("act", "none"))
