"""The work that programs give this framework, as cases that can be timed and compared.

Every case is one linear layer's GEMM, called as a serving engine or a training loop calls
it: the weight (and its scales) laid out once, an activation that is new, one call.

    linear     torch.ops.hk_vllm.linear's body: an engine's bf16 layers at decode batches
    template   hk.templates.gemm with a ready-made epilogue, bf16 operands
    gate_up    hk.templates.gemm with silu_and_mul over a merged gate and up weight
    traced     hk.templates.gemm with a program's own epilogue (squared ReLU of acc + bias)
    scaled     hk.ops.scaled_mm: fp8 e4m3, a scale a token and a scale an output channel
    wgrad      hk.ops.scaled_mm(accumulate=True): a weight gradient added to its fp32 sum,
               the e5m2 output gradient against the e4m3 activation
    mx         hk.ops.mxfp8: the activation quantized (fp8 and E8M0 scales), then the GEMM
"""

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "hk-dsl_amd"))

import hk  # noqa: E402
from hk.integration import vllm_gemm  # noqa: E402

gemm = hk.templates.gemm
E4M3, E5M2 = torch.float8_e4m3fn, torch.float8_e5m2

#: (N, K) of the linear layers of the two models the engine's route table is measured on, LM
#: heads left out: qkv, o, gate_up and down of each.
LAYERS = ((6144, 4096), (4096, 4096), (24576, 4096), (4096, 12288), (28672, 4096), (4096, 14336))
#: (N, K) of the block-scaled layers of the MX route table.
MX_LAYERS = ((1792, 5120), (2304, 5120), (5120, 1152), (5120, 4096), (16384, 1280),
             (12800, 6144), (4096, 1280))


def squared_relu(acc, ctx):
    """relu(acc + bias)^2, an MLP activation that a program writes for itself."""
    acc = (acc + ctx.bias).relu()
    return acc * acc


EPILOGUES = {"none": None, "bias": gemm.bias, "bias_gelu": gemm.bias_gelu,
             "bias_silu": gemm.bias_silu, "residual": gemm.residual,
             "bias_residual": gemm.bias_residual, "scale": gemm.scale}


def listed():
    return [
        # one token through an engine's attention output projection: the smallest call
        dict(name="linear_o_1", kind="linear", m=1, n=4096, k=4096, bias=False),
        # a small MLP's first layer at a short batch: launches and latency count
        dict(name="bias_gelu_small", kind="template", m=256, n=1024, k=1024,
             epilogue="bias_gelu", out="bfloat16"),
        # the MLP's gate and up projection of a decode batch of 16
        dict(name="gate_up_decode_16", kind="gate_up", m=16, n=24576, k=4096),
        # the same of a prefill chunk
        dict(name="gate_up_prefill_2048", kind="gate_up", m=2048, n=24576, k=4096),
        # an up projection with bias and GELU over a long prefill
        dict(name="bias_gelu_prefill_4096", kind="template", m=4096, n=12288, k=4096,
             epilogue="bias_gelu", out="bfloat16"),
        # a down projection with bias and residual on a ragged chunk of tokens
        dict(name="bias_residual_ragged_333", kind="template", m=333, n=4096, k=14336,
             epilogue="bias_residual", out="bfloat16"),
        # an fp8 qkv projection with its bias at a decode batch
        dict(name="scaled_decode_8", kind="scaled", m=8, n=6144, k=4096, bias=True),
        # an fp8 layer with bias over a long prefill
        dict(name="scaled_prefill_8192", kind="scaled", m=8192, n=4096, k=4096, bias=True),
        # a block-scaled layer at a decode batch
        dict(name="mx_decode_32", kind="mx", m=32, n=5120, k=4096),
        # the same over a prefill
        dict(name="mx_prefill_4096", kind="mx", m=4096, n=5120, k=4096),
        # the backward pass of a square layer: its weight gradient over 8192 tokens
        dict(name="wgrad_8192", kind="wgrad", m=4096, n=4096, k=8192),
        # a program's own activation on an up projection
        dict(name="traced_relu2_1024", kind="traced", m=1024, n=12288, k=4096),
    ]


def _log(rng, lo, hi, step=1):
    """A whole multiple of `step` from lo to hi, even over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(("linear", "template", "template", "gate_up", "traced", "scaled",
                       "scaled", "wgrad", "mx", "mx"))
    if kind == "linear":
        n, k = rng.choice(LAYERS)
        return dict(kind=kind, m=_log(rng, 1, 32), n=n, k=k, bias=rng.random() < 0.5)
    if kind == "template":
        # K of 64 and up in 64s, N in 4s: what the template takes
        m, k = _log(rng, 1, 4096), _log(rng, 256, 14336, 64)
        n = _log(rng, 256, 12288, rng.choice((4, 8, 64, 128)))
        out = rng.choice(("bfloat16", "bfloat16", "bfloat16", "float16", "float32",
                          "float8_e4m3fn", "int8"))
        e = "scale" if out in ("float8_e4m3fn", "int8") else rng.choice(
            [x for x in EPILOGUES if x != "scale"])
        return _within(dict(kind=kind, m=m, n=n, k=k, epilogue=e, out=out))
    if kind == "gate_up":
        # M a decode batch or a prefill chunk; 2 N' rows of gate and up
        return _within(dict(kind=kind, m=_log(rng, 1, 4096),
                            n=2 * _log(rng, 512, 14336, rng.choice((8, 64, 128))),
                            k=_log(rng, 512, 8192, rng.choice((128, 1024)))))
    if kind == "traced":
        return _within(dict(kind=kind, m=_log(rng, 1, 4096),
                            n=_log(rng, 256, 12288, rng.choice((4, 64, 128))),
                            k=_log(rng, 256, 8192, 64)), 2e11)
    if kind == "scaled":
        return _within(dict(kind=kind, m=_log(rng, 1, 8192),
                            n=_log(rng, 256, 12288, rng.choice((4, 8, 128))),
                            k=_log(rng, 256, 14336, rng.choice((128, 512))),
                            bias=rng.random() < 0.5))
    if kind == "wgrad":
        return _within(dict(kind=kind, m=_log(rng, 512, 8192, 8), n=_log(rng, 512, 8192, 8),
                            k=_log(rng, 512, 16384, 128)), 2.7e11)
    n, k = rng.choice(MX_LAYERS)
    if rng.random() < 0.5:  # a layer of the same ranges that the table does not hold
        n, k = _log(rng, 512, 12800, 8), _log(rng, 512, 6144, 128)
    return _within(dict(kind="mx", m=_log(rng, 1, 8192), n=n, k=k), 2.7e11)


def _within(case, flops=4.1e11):
    """The case with M cut so that it costs no more than the largest listed one."""
    most = int(flops / (2 * case["n"] * case["k"]))
    if case["m"] > most:
        case["m"] = most // 8 * 8 if case["kind"] == "wgrad" else most
    return case


# ---------------------------------------------------------------- inputs


def _inputs(case, seed):
    """The call's inputs on the GPU, from the seed alone: x ~ N(0, 1), weights ~ N(0, 0.02),
    biases ~ N(0, 0.1); fp8 operands are such tensors scaled to the format's range."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, m, n, k = case["kind"], case["m"], case["n"], case["k"]

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * std

    if kind == "wgrad":
        # the gradient's last axis is tokens: (out, tokens) and (in, tokens)
        dy, x = normal(m, k, std=1e-3), normal(n, k)
        sa, sb = dy.abs().amax() / 57344, x.abs().amax() / 448
        return dict(a=(dy / sa).to(E5M2), b=(x / sb).to(E4M3), sa=sa.reshape(1),
                    sb=sb.reshape(1), grad=normal(m, n, std=0.1))
    x, w = normal(m, k), normal(n, k, std=0.02)
    if kind == "scaled":
        sa = x.abs().amax(1, keepdim=True) / 448
        sb = w.abs().amax(1) / 448
        return dict(a=(x / sa).to(E4M3), b=(w / sb[:, None]).to(E4M3), sa=sa, sb=sb,
                    bias=normal(n, std=0.1).bfloat16() if case["bias"] else None)
    if kind == "mx":
        wq, ws = _mx_quant(w)
        return dict(x=x.bfloat16(), w=wq, ws=ws)
    s = dict(x=x.bfloat16(), w=w.bfloat16())
    if kind == "linear":
        s["bias"] = normal(n, std=0.1).bfloat16() if case["bias"] else None
    elif kind == "traced":
        s["bias"] = normal(n, std=0.1).bfloat16()
    elif kind == "template":
        e = case["epilogue"]
        ops = s["ops"] = {}
        if "bias" in e:
            ops["bias"] = normal(n, std=0.1).bfloat16()
        if "residual" in e:
            ops["residual"] = normal(m, n).bfloat16()
        if e == "scale":  # a quantizer: a scale an output channel, C's spread within range
            top = 448.0 if case["out"] == "float8_e4m3fn" else 127.0
            spread = 4.5 * 0.02 * math.sqrt(k)
            ops["scale"] = top / spread * (0.5 + torch.rand(n, generator=g, device="cuda"))
    return s


def _mx_quant(w):
    """A checkpoint's block-scaled weight: fp8 rows with an E8M0 scale every 32 columns."""
    e = _mx_exponent(w)
    q = (w.reshape(w.shape[0], -1, 32) * torch.exp2(-e)[..., None]).clamp(-448, 448)
    return q.reshape(w.shape).to(E4M3), (e + 127).to(torch.uint8)


def _mx_exponent(x):
    """The smallest whole e with max |x| <= 448 * 2^e for each 32 values of a row."""
    amax = x.reshape(x.shape[0], -1, 32).abs().amax(2).clamp(min=2.0 ** -126)
    mant, exp = torch.frexp(amax)  # amax = mant * 2^exp, mant in [0.5, 1); 448 = 0.875 * 2^9
    return (exp - 9 + (mant > 0.875)).to(x.dtype)


def prepare(case, seed):
    return dict(_inputs(case, seed), case=case)


# ---------------------------------------------------------------- the call


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return vllm_gemm.linear(state["x"], state["w"], state["bias"])
    if kind == "template":
        return gemm(state["x"], state["w"], epilogue=EPILOGUES[case["epilogue"]],
                    out_dtype=getattr(torch, case["out"]), **state["ops"])
    if kind == "gate_up":
        return gemm(state["x"], state["w"], epilogue=gemm.silu_and_mul)
    if kind == "traced":
        return gemm(state["x"], state["w"], epilogue=squared_relu, bias=state["bias"])
    if kind == "scaled":
        return hk.ops.scaled_mm(state["a"], state["b"], state["sa"], state["sb"],
                                bias=state["bias"])
    if kind == "wgrad":
        return hk.ops.scaled_mm(state["a"], state["b"], state["sa"], state["sb"],
                                out=state["grad"], accumulate=True)
    q, s = hk.ops.mxfp8.quant(state["x"])
    return q, s, hk.ops.mxfp8.gemm(q, state["w"], s, state["ws"])


# ---------------------------------------------------------------- what it costs


def work(case):
    kind, m, n, k = case["kind"], case["m"], case["n"], case["k"]
    flops = 2 * m * n * k
    if kind == "wgrad":
        return {"bytes": (m + n) * k + 8 * m * n, "flops": flops}
    if kind == "scaled":
        return {"bytes": (m + n) * k + 2 * m * n + 4 * (m + n) + 2 * n * case["bias"],
                "flops": flops}
    if kind == "mx":  # x read, q and its scales written; w and its scales read, y written
        return {"bytes": 2 * m * k + (m + n) * (k + k // 32) + 2 * m * n, "flops": flops}
    nbytes = 2 * (m + n) * k
    if kind == "gate_up":
        return {"bytes": nbytes + m * n, "flops": flops}
    if kind == "template":
        e, ob = case["epilogue"], getattr(torch, case["out"]).itemsize
        nbytes += ob * m * n + 2 * n * ("bias" in e) + 2 * m * n * ("residual" in e)
        return {"bytes": nbytes + 4 * n * (e == "scale"), "flops": flops}
    return {"bytes": nbytes + 2 * m * n + 2 * n * (kind == "traced" or bool(case["bias"])),
            "flops": flops}


def tolerance(case):
    """bf16 outputs of fp32 sums differ by the last bit of a few values; the same for the
    other types of C, whose last bit is larger or smaller."""
    out = {"wgrad": "float32", "template": case.get("out")}.get(case["kind"], "bfloat16")
    return {"float32": {"rel": 3e-5, "max": 3e-4},
            "float16": {"rel": 1e-3, "max": 3e-3},
            "bfloat16": {"rel": 6e-3, "max": 2e-2},
            "float8_e4m3fn": {"rel": 6e-3, "max": 0.15},
            "int8": {"differ": 1e-3}}[out]


# ---------------------------------------------------------------- 64 bits


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]

    def d(t):
        return t.float().double()

    if kind == "wgrad":
        return d(s["grad"]) + (d(s["a"]) @ d(s["b"]).t()) * d(s["sa"]) * d(s["sb"])
    if kind == "scaled":
        y = (d(s["a"]) @ d(s["b"]).t()) * d(s["sa"]) * d(s["sb"])
        return y if s["bias"] is None else y + d(s["bias"])
    if kind == "mx":
        x = d(s["x"])
        e = _mx_exponent(x)
        q = (x.reshape(x.shape[0], -1, 32) * torch.exp2(-e)[..., None]).clamp(-448, 448)
        q = d(q.float().to(E4M3))
        w = d(s["w"]).reshape(s["w"].shape[0], -1, 32) * torch.exp2(d(s["ws"]) - 127)[..., None]
        y = (q * torch.exp2(e)[..., None]).reshape(x.shape) @ w.reshape(s["w"].shape).t()
        return q.reshape(x.shape), None, y
    y = d(s["x"]) @ d(s["w"]).t()
    if kind == "gate_up":
        gate, up = y.chunk(2, dim=1)
        return gate * torch.sigmoid(gate) * up
    if kind == "traced":
        return (y + d(s["bias"])).relu().square()
    if kind == "linear":
        return y if s["bias"] is None else y + d(s["bias"])
    ops, e = s["ops"], case["epilogue"]
    if case["out"] == "int8":
        return None
    for v in ("bias", "residual"):
        if v in ops:
            y = y + d(ops[v])
    if e == "bias_gelu":
        return torch.nn.functional.gelu(y, approximate="tanh")
    if e == "bias_silu":
        return torch.nn.functional.silu(y)
    if e == "scale":
        y = (y * d(ops["scale"])).clamp(-448, 448)
    return y
