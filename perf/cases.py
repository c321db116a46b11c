"""The quantized-linear work that a user of this package has it do, as cases to be timed.

A case is a call (or the two or three calls that a decoder's sublayer makes) of the public operators
on one layer's weights, from the smallest decode step to a long prefill, plus the load-time packing of
a layer. ``listed()`` holds the fixed cases, ``draw(rng)`` gives others of the same ranges.

Kinds:

* ``linear``: ``w4a16_linear`` / ``_residual`` / ``_silu_mul`` (``epilogue``), fp16 activations;
* ``norm_linear``: ``rmsnorm_fp8_w4a16_linear``, the sublayer input norm and its linear;
* ``mlp``: the MLP sublayer, ``norm_linear`` with SiLU*mul (gate_up) and then the residual linear (down);
* ``w4a8``: ``rmsnorm_fp8_quant`` and ``w4a8_linear`` on its codes;
* ``norm``: ``rmsnorm_fp8_quant_dequant``;
* ``pack``: ``pack_awq``, one layer's load-time conversion.

``m`` counts rows (tokens), ``n`` x ``k`` is the layer (for ``mlp``: gate_up, whose down projection is
``k`` x ``n / 2``), ``group`` the quantization group.
"""

from __future__ import annotations

import math

import torch

import tokenforge.kernels.ops  # noqa: F401  (registers torch.ops.tokenforge)
from tokenforge.kernels import pack

EPS = 1e-6

# (n, k) of the four linears of the two decoders that the numerics suite and the benchmark use.
QWEN25_7B = {"qkv": (4608, 3584), "o": (3584, 3584), "gate_up": (37888, 3584), "down": (3584, 18944)}
QWEN25_05B = {"qkv": (1152, 896), "o": (896, 896), "gate_up": (9728, 896), "down": (896, 4864)}


def _case(name, kind, m, nk, epilogue="none", bias=False, group=128):
    return {"name": name, "kind": kind, "m": m, "n": nk[0], "k": nk[1], "epilogue": epilogue, "bias": bias,
            "group": group}


def listed():
    return [
        # One decode step of a small decoder, three sequences: launch and latency, hardly any data.
        _case("small_o_m3", "linear", 3, QWEN25_05B["o"], "residual"),
        # Single-sequence decode: input norm + fused QKV projection with its bias.
        _case("decode_qkv_m1", "norm_linear", 1, QWEN25_7B["qkv"], bias=True),
        # Single-sequence decode: the whole MLP sublayer, three quarters of a decoder's weight bytes.
        _case("decode_mlp_m1", "mlp", 1, QWEN25_7B["gate_up"], "silu_mul"),
        # A handful of sequences: the longest reduction, an odd number of rows.
        _case("batch_down_m7", "linear", 7, QWEN25_7B["down"], "residual"),
        # A serving batch of some dozens of sequences.
        _case("batch_gate_up_m48", "linear", 48, QWEN25_7B["gate_up"], "silu_mul"),
        # A short prompt through a small decoder quantized in groups of 64.
        _case("small_gate_up_m333", "linear", 333, QWEN25_05B["gate_up"], "silu_mul", group=64),
        # A short prompt, or one chunk of a chunked prefill.
        _case("prefill_gate_up_m256", "linear", 256, QWEN25_7B["gate_up"], "silu_mul"),
        # A prompt of ordinary, odd length.
        _case("prefill_down_m1000", "linear", 1000, QWEN25_7B["down"], "residual"),
        # A long prompt: the largest product.
        _case("prefill_gate_up_m4096", "linear", 4096, QWEN25_7B["gate_up"], "silu_mul"),
        # The W4A8 form of the same sublayer input: norm, FP8 codes, the linear on the codes.
        _case("w4a8_gate_up_m2048", "w4a8", 2048, QWEN25_7B["gate_up"], "silu_mul"),
        # The norm of a long prompt, codes and the activation that a W4A16 linear reads.
        _case("norm_t4095", "norm", 4095, (0, 3584)),
        # Loading a checkpoint: one large layer into the kernels' layout.
        _case("load_gate_up", "pack", 0, QWEN25_7B["gate_up"]),
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choices(("linear", "norm_linear", "mlp", "w4a8", "norm", "pack"), (10, 2, 2, 3, 2, 2))[0]
    group = rng.choices((128, 64, 32), (8, 2, 1))[0]
    epilogue = rng.choice(("none", "residual", "silu_mul")) if kind in ("linear", "w4a8") else (
        rng.choice(("none", "silu_mul")) if kind == "norm_linear" else "silu_mul" if kind == "mlp" else "none")
    if kind == "norm":
        return _norm_draw(rng)
    decoder = rng.choice((QWEN25_7B, QWEN25_05B, None))
    if kind == "mlp":
        n, k = (decoder or QWEN25_05B)["gate_up"]
    elif decoder is not None:
        n, k = decoder[rng.choice(("gate_up",) if epilogue == "silu_mul" else ("qkv", "o", "gate_up", "down"))]
    else:  # a layer of some other decoder, now and then with an N that no tile divides
        n = _log_int(rng, 256, 32768, 16 if epilogue == "silu_mul" or rng.random() < 0.7 else 8)
        k = _log_int(rng, 256, 16384, 128)
    m = _log_int(rng, 1, 4096)
    if kind == "norm_linear":
        k, m = min(k, 8192), min(m, 2048)
    if kind == "mlp":
        m = min(m, 2048)
    if kind == "pack":
        m = 0
    m = min(m, 4096 * 37888 * 3584 // (n * k))
    c = _case("", kind, m, (n, k), epilogue, rng.random() < 0.3 and kind in ("linear", "norm_linear"), group)
    del c["name"]
    return c


def _norm_draw(rng):
    c = _case("", "norm", _log_int(rng, 64, 8192), (0, rng.choice((896, 1024, 2048, 3584, 4096, 5120, 8192))))
    del c["name"]
    return c


# ----------------------------------------------------------------------------- inputs


def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed))


def _nibbles(n, k, group, gen):
    """4-bit weights and zero points as min-max quantization of a roughly normal weight gives them:
    codes bell-shaped over 0..15, zero points around the middle; scales a few thousandths."""
    dev = gen.device
    q = (torch.randn((k, n), generator=gen, device=dev, dtype=torch.float16) * 2.8 + 7.5).round().clamp(0, 15)
    z = (torch.randn((k // group, n), generator=gen, device=dev) + 7.5).round().clamp(0, 15)
    s = (torch.rand((k // group, n), generator=gen, device=dev) * 4e-3 + 4e-3).to(torch.float16)
    return q.to(torch.uint8), z.to(torch.uint8), s


def _awq_words(v):
    """[rows, n] values 0..15 -> int32 [rows, n / 8]: offsets 0 2 4 6 1 3 5 7 in nibbles 0..7."""
    v = v.reshape(v.shape[0], -1, 8)
    out = torch.zeros(v.shape[:2], dtype=torch.int32, device=v.device)
    for nib, off in enumerate((0, 2, 4, 6, 1, 3, 5, 7)):
        out |= v[:, :, off].to(torch.int32) << (4 * nib)
    return out


def _awq(n, k, group, gen):
    q, z, s = _nibbles(n, k, group, gen)
    return _awq_words(q), _awq_words(z), s


def _inputs(case, seed):
    """Everything that is drawn for a case, in one order: the same values for prepare and exact."""
    gen = _gen(seed)
    m, n, k = case["m"], case["n"], case["k"]
    h = lambda *shape: torch.randn(shape, generator=gen, device="cuda").to(torch.float16)  # noqa: E731
    d = {"gen": gen}
    if case["kind"] != "pack":
        d["x"] = h(m, k)
    if case["kind"] in ("norm", "norm_linear", "mlp", "w4a8"):
        d["gamma"] = (1 + 0.1 * h(k)).to(torch.float16)
    if case["bias"]:
        d["bias"] = (0.1 * h(n)).to(torch.float16)
    if case["epilogue"] == "residual":
        d["residual"] = h(m, n)
    return d


def prepare(case, seed):
    s = {"case": case, "g": case["group"], **_inputs(case, seed)}
    gen = s.pop("gen")
    n, k, g = case["n"], case["k"], case["group"]
    if case["kind"] == "norm":
        return s
    awq = _awq(n, k, g, gen)
    if case["kind"] == "pack":
        s["awq"] = awq
        return s
    s["w"] = pack.pack_awq(awq[0], awq[1], awq[2], g)
    if case["kind"] == "mlp":
        awq = _awq(k, n // 2, g, gen)
        s["w2"] = pack.pack_awq(awq[0], awq[1], awq[2], g)
    return s


# ----------------------------------------------------------------------------- one pass


def run(s):
    case, g = s["case"], s["g"]
    kind, epi = case["kind"], case["epilogue"]
    ops = torch.ops.tokenforge
    if kind == "pack":
        w = pack.pack_awq(s["awq"][0], s["awq"][1], s["awq"][2], g)
        return w.qweight_t, w.scales, w.qzeros
    x = s["x"]
    if kind == "norm":
        q, scale, a = ops.rmsnorm_fp8_quant_dequant(x, s["gamma"], EPS, None)
        return q.view(torch.uint8), scale, a
    w, bias = s["w"], s.get("bias")
    if kind == "norm_linear":
        return ops.rmsnorm_fp8_w4a16_linear(x, s["gamma"], EPS, w.qweight_t, w.scales, w.qzeros, bias, g, "hip", epi)
    if kind == "mlp":
        act = ops.rmsnorm_fp8_w4a16_linear(x, s["gamma"], EPS, w.qweight_t, w.scales, w.qzeros, None, g, "hip",
                                           "silu_mul")
        w2 = s["w2"]
        return ops.w4a16_linear_residual(act, w2.qweight_t, w2.scales, w2.qzeros, None, x, g, "hip")
    if kind == "w4a8":
        q, scale = ops.rmsnorm_fp8_quant(x, s["gamma"], EPS, None)
        y = ops.w4a8_linear(q, scale, w.qweight_t, w.scales, w.qzeros, None, g, "hip", epi, s.get("residual"))
        return q.view(torch.uint8), scale, y
    if epi == "residual":
        return ops.w4a16_linear_residual(x, w.qweight_t, w.scales, w.qzeros, bias, s["residual"], g, "hip")
    if epi == "silu_mul":
        return ops.w4a16_linear_silu_mul(x, w.qweight_t, w.scales, w.qzeros, bias, g, "hip")
    return ops.w4a16_linear(x, w.qweight_t, w.scales, w.qzeros, bias, g, "hip")


# ----------------------------------------------------------------------------- what a pass needs


def _weight_bytes(n, k, g):
    return n * k // 2 + (k // g) * n * 2 + (k // g) * n // 2


def work(case):
    m, n, k, g, kind = case["m"], case["n"], case["k"], case["group"], case["kind"]
    if kind == "pack":
        return {"bytes": 2 * _weight_bytes(n, k, g), "flops": 0}
    if kind == "norm":
        return {"bytes": m * k * 2 + k * 2 + m * k + m * 4 + m * k * 2, "flops": 0}
    if kind == "mlp":
        return {"bytes": _weight_bytes(n, k, g) + _weight_bytes(k, n // 2, g) + k * 2 + 2 * m * k * 2,
                "flops": 2 * m * n * k + m * n * k}
    n_out = n // 2 if case["epilogue"] == "silu_mul" else n
    b = _weight_bytes(n, k, g) + m * k * 2 + m * n_out * 2
    if case["epilogue"] == "residual":
        b += m * n * 2
    if case["bias"]:
        b += n * 2
    if kind in ("norm_linear", "w4a8"):
        b += k * 2
    if kind == "w4a8":  # the codes and their scales are results too
        b += m * k + m * 4
    return {"bytes": b, "flops": 2 * m * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind == "pack":
        return "exact"
    if kind == "norm":  # an e4m3 rounding may fall the other way on a code in a thousand
        return {"rel": 2e-3, "max": 0.15, "differ": 1e-3}
    if kind in ("norm_linear", "mlp", "w4a8"):  # ... and the product follows it
        return {"rel": 2e-3, "max": 0.05, "differ": 1e-3}
    # fp32 sums in another order, rounded to fp16 (SiLU*mul: three roundings)
    return {"rel": 1.5e-3 if case["epilogue"] == "silu_mul" else 1e-3, "max": 0.02}


# ----------------------------------------------------------------------------- 64 bits


def _dense64(n, k, g, gen, fp16_weights):
    q, z, s = _nibbles(n, k, g, gen)
    w = torch.empty((n, k), dtype=torch.float64, device=q.device)
    step = max(1, (1 << 24) // n) * g  # rows of K at a time
    for a in range(0, k, step):
        b = min(k, a + step)
        grp = torch.arange(a, b, device=q.device) // g
        d = (q[a:b].to(torch.int16) - z[grp].to(torch.int16))
        part = (d.to(torch.float16) * s[grp]).double() if fp16_weights else d.double() * s[grp].double()
        w[:, a:b] = part.t()
    return w


def _norm64(x, gamma):
    """(codes as fp64 values, scales [rows, 1]) of the RMSNorm and its dynamic e4m3 quantization."""
    x = x.double()
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()
    scale = torch.clamp(y.abs().amax(-1, keepdim=True) / 448.0, min=1.0 / (448.0 * 512.0))
    v = (y / scale).clamp(-448.0, 448.0)
    return v.float().to(torch.float8_e4m3fn).double(), scale


def _finish64(case, y, d):
    n = case["n"]
    if "bias" in d:
        y = y + d["bias"].double()
    if case["epilogue"] == "silu_mul":
        return torch.nn.functional.silu(y[:, : n // 2]) * y[:, n // 2:]
    return y + d["residual"].double() if case["epilogue"] == "residual" else y


def exact(case, seed):
    kind = case["kind"]
    if kind == "pack":
        return None
    d = _inputs(case, seed)
    n, k, g = case["n"], case["k"], case["group"]
    if kind == "linear":
        return _finish64(case, d["x"].double() @ _dense64(n, k, g, d["gen"], True).t(), d)
    code, scale = _norm64(d["x"], d["gamma"])
    if kind == "norm":
        return None, scale, code * scale
    y = _finish64(case, (code * scale) @ _dense64(n, k, g, d["gen"], kind != "w4a8").t(), d)
    if kind == "w4a8":
        return None, scale, y
    if kind == "mlp":
        return d["x"].double() + y @ _dense64(k, n // 2, g, d["gen"], True).t()
    return y
