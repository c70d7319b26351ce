"""The work that users of this framework have it do, as measurable cases: one expert layer of a mixture-of-experts
model, called the way a model's program calls it - `GLUMLP` / `MLP`, or the Hugging Face injection
(`experts_forward`, `gpt_oss_forward`) - from one decoded token to a training step over tens of thousands.

A case is a dict of
  module    "glu" (GLUMLP, SiLU), "mlp" (MLP, GELU), "hf" (experts_forward: act(gate) * up, weights (E, out, in)),
            "oss" (gpt_oss_forward: clamped gated unit, biases, weights (E, in, out))
  train     False: forward under no_grad; True: forward and backward, every gradient
  router    True: the routing comes from (T, E) logits through `topk_softmax`, as in the Granite injection;
            False: the caller already holds the (T, k) routing weights and expert ids
  dtype, T (tokens), d (model width), f (expert width), E (experts), k (experts per token), bias,
  skew      0: evenly spread routing; b: logits shifted by -1.2 b log(rank), the Zipf-like load of a router that
            has not been balanced
"""
import math

import torch
from torch import nn

from scattermoe_amd.kernels import ops
from scattermoe_amd.mlp import GLUMLP, MLP
from scattermoe_amd.utils import replace_moe

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda:0"

# Expert shapes of the benchmark's workloads: Mixtral-like, gpt-oss-like and fine-grained (Qwen-like)
WIDE = {"d": 4096, "f": 14336, "E": 8, "k": 2}
SQUARE = {"d": 2880, "f": 2880, "E": 32, "k": 4}
FINE = {"d": 2048, "f": 768, "E": 128, "k": 8}


def _case(name, shape, T, module="glu", train=False, dtype="bf16", bias=False, skew=0.0, router=False):
    return dict(shape, name=name, T=T, module=module, train=train, dtype=dtype, bias=bias, skew=skew, router=router)


def listed():
    return [
        # one token of one user: the latency of a decode step, fine-grained experts (75 MB of weights touched)
        _case("decode_1_fine", FINE, 1),
        # the same with the widest experts (705 MB of weights: a pure stream)
        _case("decode_1_wide", WIDE, 1),
        # serving: a batch of sequences decodes one token each; every expert gets a few rows
        _case("decode_48_oss", SQUARE, 48, module="oss", bias=True),
        _case("decode_64_wide", WIDE, 64),
        # a larger serving batch over many experts
        _case("decode_200_fine", FINE, 200),
        # a prompt of ordinary, ragged length through the Hugging Face injection in half precision
        _case("prefill_777_hf_fp16", WIDE, 777, module="hf", dtype="fp16"),
        # a long prompt, routed from router logits
        _case("prefill_3999_fine", FINE, 3999, router=True),
        # a toy model in full precision (the size of a unit test or of a research prototype): launches and host work
        _case("train_256_fp32", {"d": 128, "f": 256, "E": 8, "k": 2}, 256, module="mlp", train=True, dtype="fp32"),
        # fine-tuning through the Hugging Face injection on a short, ragged batch
        _case("train_1501_oss", SQUARE, 1501, module="oss", train=True, bias=True),
        # pre-training steps of the benchmark's workloads
        _case("train_8192_skewed", SQUARE, 8192, train=True, bias=True, skew=1.5),
        _case("train_32768_fine", FINE, 32768, train=True),
        _case("train_16384_wide", WIDE, 16384, train=True),
    ]


# what the largest listed case costs; nothing drawn goes beyond it
MOST_ROWS = 262144
MOST_ROW_PRODUCTS = 32768 * 4096 * 14336        # rows * d * f
MOST_PARAMETERS = 3 * 8 * 4096 * 14336


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    family = rng.choices(("decode", "prefill", "train", "fp32"), (6, 5, 7, 2))[0]
    if family == "fp32":
        # the grid of the module tests: odd widths, some of them not a whole number of 16-byte pieces
        d, k = rng.choice((100, 128, 256, 512, 600)), rng.choice((2, 3, 4))
        return {"d": d, "f": 4 * d // k, "E": 8, "k": k, "T": int(_log_uniform(rng, 32, 2048)), "module": "mlp",
                "train": rng.random() < 0.7, "dtype": "fp32", "bias": rng.random() < 0.5, "skew": 0.0,
                "router": False}
    if rng.random() < 0.5:
        shape = dict(rng.choice((WIDE, SQUARE, FINE)))
    else:
        step = 64 if rng.random() < 0.7 else 8
        E = rng.choice((8, 16, 32, 64, 128))
        shape = {"d": round(_log_uniform(rng, 256, 4096) / step) * step,
                 "f": round(_log_uniform(rng, 256, 14336) / step) * step,
                 "E": E, "k": rng.choice([k for k in (1, 2, 4, 6, 8) if 2 * k <= E])}
        while 3 * shape["E"] * shape["d"] * shape["f"] > MOST_PARAMETERS:
            shape["f"] = round(shape["f"] / 2 / step) * step
    module = rng.choices(("glu", "hf", "oss", "mlp"), (5, 2, 3, 1))[0]
    lo, hi = {"decode": (1, 512), "prefill": (256, 16384), "train": (256, 32768)}[family]
    T = int(_log_uniform(rng, lo, hi + 1))
    train = family == "train"
    rows = MOST_ROW_PRODUCTS * (1 if train else 3) / (shape["d"] * shape["f"])
    T = max(1, min(T, int(min(rows, MOST_ROWS) / shape["k"])))
    return dict(shape, T=T, module=module, train=train, dtype=rng.choices(("bf16", "fp16"), (3, 1))[0],
                bias=module == "oss" or (module != "hf" and rng.random() < 0.3),
                skew=rng.choice((0.0, 0.0, 0.7, 1.5)), router=shape["k"] > 1 and rng.random() < 0.25)


class _HFExperts(nn.Module):
    """The attributes that `experts_forward` finds on a Hugging Face experts module."""

    def __init__(self, d, f, E):
        super().__init__()
        self.num_experts = E
        self.gate_up_proj = nn.Parameter(torch.empty(E, 2 * f, d))
        self.down_proj = nn.Parameter(torch.empty(E, d, f))
        self.act_fn = nn.SiLU()


class _OssExperts(nn.Module):
    """The attributes that `gpt_oss_forward` finds on a gpt-oss experts module."""

    def __init__(self, d, f, E):
        super().__init__()
        self.hidden_size, self.num_experts, self.alpha, self.limit = d, E, 1.702, 7.0
        self.gate_up_proj = nn.Parameter(torch.empty(E, d, 2 * f))
        self.gate_up_proj_bias = nn.Parameter(torch.empty(E, 2 * f))
        self.down_proj = nn.Parameter(torch.empty(E, f, d))
        self.down_proj_bias = nn.Parameter(torch.empty(E, d))


def _module(case, dtype):
    d, f, E, k = (case[n] for n in ("d", "f", "E", "k"))
    if case["module"] == "glu":
        return GLUMLP(d, f, E, k, bias=case["bias"]).to(dtype)
    if case["module"] == "mlp":
        return MLP(d, f, E, k, bias=case["bias"], activation=nn.GELU()).to(dtype)
    return (_HFExperts if case["module"] == "hf" else _OssExperts)(d, f, E).to(dtype)


def prepare(case, seed):
    """Weights N(0, 0.02) as the modules initialise them, token rows and output gradients N(0, 1), routing from
    random router logits (softmax, top-k, renormalised)."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype, T, E, k = DTYPES[case["dtype"]], case["T"], case["E"], case["k"]
    with torch.device("meta"):
        module = _module(case, dtype)
    module = module.to_empty(device=DEVICE)
    with torch.no_grad():
        for p in module.parameters():
            p.normal_(0.0, 0.02, generator=g)
    logits = torch.randn(T, E, generator=g, device=DEVICE)
    if case["skew"]:
        logits -= 1.2 * case["skew"] * torch.log(torch.arange(1, E + 1, device=DEVICE, dtype=torch.float32))
    x = torch.randn(T, case["d"], generator=g, device=DEVICE, dtype=dtype)
    state = {"case": case, "module": module, "x": x, "logits": None, "gates": None, "experts": None}
    if case["router"]:
        state["logits"] = logits.to(dtype)
    else:
        gates, experts = torch.topk(torch.softmax(logits, -1), k)
        state["gates"] = (gates / gates.sum(-1, keepdim=True)).to(dtype)
        state["experts"] = experts
    if case["train"]:
        state["dy"] = torch.randn(T, case["d"], generator=g, device=DEVICE, dtype=dtype)
        source = state["logits"] if case["router"] else state["gates"]
        state["leaves"] = [x.requires_grad_(), source.requires_grad_()] + list(module.parameters())
    return state


def _forward(s):
    case, x, gates, experts = s["case"], s["x"], s["gates"], s["experts"]
    if case["router"]:
        gates, experts = ops.topk_softmax(s["logits"], case["k"])
        gates = gates.to(x.dtype)
    if case["module"] == "oss":
        return replace_moe.gpt_oss_forward(s["module"], x, experts, gates)
    if case["module"] == "hf":
        return replace_moe.experts_forward(s["module"], x, experts, gates)
    return s["module"](x, gates, experts)


def run(s):
    if not s["case"]["train"]:
        with torch.no_grad():
            return _forward(s)
    for t in s["leaves"]:
        t.grad = None
    y = _forward(s)
    y.backward(s["dy"])
    return [y.detach()] + [t.grad for t in s["leaves"]]


def work(case):
    """Weights of the experts that are hit (training: read, and every weight's gradient written), token rows in and
    out, routing; the products of the two layers (training: each of them three times)."""
    T, d, f, E, k = (case[n] for n in ("T", "d", "f", "E", "k"))
    size = 4 if case["dtype"] == "fp32" else 2
    n1 = f if case["module"] == "mlp" else 2 * f
    per_expert = (n1 + f) * d + (n1 + d if case["bias"] else 0)
    p = [1.0] * E
    if case["skew"]:
        p = [(r + 1) ** (-1.2 * case["skew"]) for r in range(E)]
    total = sum(p)
    hit = sum(1.0 - max(0.0, 1.0 - min(1.0, k * q / total)) ** T for q in p)
    routing = T * E * size if case["router"] else T * k * (size + 8)
    flops = 2.0 * T * k * d * (n1 + f)
    if not case["train"]:
        return {"bytes": hit * per_expert * size + 2 * T * d * size + routing, "flops": flops}
    return {"bytes": (hit + E) * per_expert * size + 4 * T * d * size + 2 * routing, "flops": 3 * flops}


def tolerance(case):
    """About four times what the same path gives with both of its contractions in another order (model width and
    hidden units permuted), worst output over the listed and thirty drawn cases: bf16 1.1e-3 (largest single value
    3.2e-2), fp16 2.5e-4 (5e-3), fp32 1.0e-6 (7e-6).  The gate gradients are the worst: dot products over stored,
    rounded rows."""
    return {"bf16": {"rel": 4.5e-3, "max": 0.13}, "fp16": {"rel": 1e-3, "max": 0.025},
            "fp32": {"rel": 4e-6, "max": 3e-5}}[case["dtype"]]
