"""The work that this package does for a program that serves a radix-packed
model, as a list of measured cases.

A case is one pass of a kind of work:

  linears  the packed Linears of one decoder block, or one of them, called as
           a serving loop calls the swapped modules (q/k/v and gate/up through
           install_groups), for m activation rows: m = 1 is a decode step,
           2..8 the verify rows of speculative decoding, more a prefill chunk
           (the weight decoded once, then F.linear)
  narrow   a raw bf16 Linear under the codec's row threshold (NarrowLinear)
  pack     the encoder: bf16 bits of one weight to its packed arrays, on the
           host, as a program that packs a checkpoint calls it

Weights are N(0, 0.02), or Student-t (nu = 4) of the same deviation, which
has more rare exponents; activations are N(0, 1) and biases N(0, 0.02).
`prepare` packs the weights and makes the modules resident, as a loader does
once; `run` is the forward calls alone.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from drinkme_amd import radix_pack, swap

# (name, rows, columns) of the Linears of a block
LAYER_8B = "q_proj:4096x4096 k_proj:1024x4096 v_proj:1024x4096 o_proj:4096x4096 " \
           "gate_proj:12288x4096 up_proj:12288x4096 down_proj:4096x12288"
MLP_32B = "gate_proj:25600x5120 up_proj:25600x5120 down_proj:5120x25600"
ATTENTION_32B = "q_proj:8192x5120 k_proj:1024x5120 v_proj:1024x5120 o_proj:5120x8192"
# columns that are not whole 1024-weight blocks: 3.5 and 9.25 of them
MLP_RAGGED = "gate_proj:9472x3584 up_proj:9472x3584 down_proj:3584x9472"

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
# bits a weight takes in the packed payload, by profile and distribution
BITS = {("sip", "normal"): 11.19, ("sip", "t4"): 11.33, ("balanced", "normal"): 10.77, ("balanced", "t4"): 10.94,
        ("gulp", "normal"): 10.74, ("gulp", "t4"): 10.87}


def _linears(name, shapes, profile, m, x="bf16", bias=False, dist="normal"):
    return {"name": name, "kind": "linears", "shapes": shapes, "profile": profile, "m": m, "x": x, "bias": bias,
            "dist": dist}


def listed():
    return [
        # the smallest call of a decode step: one k/v projection, one row
        _linears("kv-sip-m1", "k_proj:1024x4096", "sip", 1),
        # a decode step's block at the default profile: the most frequent work there is
        _linears("layer-sip-m1", LAYER_8B, "sip", 1),
        # the MLP of a larger model at the densest profile, heavy-tailed weights
        _linears("mlp-gulp-m1", MLP_32B, "gulp", 1, dist="t4"),
        # the head, the largest weight of a decode step
        _linears("head-sip-m1", "lm_head:151936x4096", "sip", 1),
        # speculative decoding: one accepted and three draft rows
        _linears("layer-gulp-m4", LAYER_8B, "gulp", 4),
        # the widest verify call, eight rows
        _linears("layer-sip-m8", LAYER_8B, "sip", 8),
        # a hidden size that is no whole number of blocks, as many models have
        _linears("ragged-sip-m1", MLP_RAGGED, "sip", 1),
        # a model that keeps its activations in fp32, with biases, two rows
        _linears("attention-gulp-f32-m2", ATTENTION_32B, "gulp", 2, x="f32", bias=True),
        # the middle profile, a decode step's attention block with q/k/v biases
        _linears("attention-balanced-m1", LAYER_8B.split(" gate")[0], "balanced", 1, bias=True),
        # a prefill chunk through an MLP of the default profile
        _linears("prefill-sip-m128", LAYER_8B.split("o_proj:4096x4096 ")[1], "sip", 128),
        # a raw Linear below the codec's row threshold (a router, a gate), four rows
        {"name": "narrow-m4", "kind": "narrow", "rows": 256, "cols": 6656, "m": 4, "x": "bf16", "bias": True},
        # packing one weight of a checkpoint
        {"name": "pack-sip", "kind": "pack", "rows": 4096, "cols": 4096, "profile": "sip", "dist": "normal"},
    ]


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, hi):
    """A column count the codec takes: whole blocks half of the time, else
    any multiple of 4."""
    c = _log_between(rng, 1024, hi)
    return max(1024, c // 1024 * 1024) if rng.random() < 0.5 else max(1024, c // 4 * 4)


def draw(rng):
    u = rng.random()
    if u < 0.1:
        return {"kind": "narrow", "rows": _log_between(rng, 16, 1023), "cols": _log_between(rng, 1024, 16384) // 4 * 4,
                "m": rng.randint(1, 8), "x": rng.choice(["bf16", "bf16", "f32"]), "bias": rng.random() < 0.5}
    profile, dist = rng.choice(["sip", "sip", "gulp", "gulp", "balanced"]), rng.choice(["normal", "normal", "t4"])
    if u < 0.15:
        return {"kind": "pack", "rows": _log_between(rng, 1024, 8192), "cols": _cols(rng, 8192), "profile": profile,
                "dist": dist}
    x = rng.choice(["bf16", "bf16", "bf16", "f32", "f16"])
    m = rng.choice([1, 1, 1, 2, 3, 4, 4, 5, 6, 7, 8])
    if u < 0.3:
        m, x = _log_between(rng, 9, 512), "bf16"
    kind = rng.choice(["one", "one", "attention", "mlp"])
    hidden = _cols(rng, 8192)
    if kind == "one":
        rows, cols = _log_between(rng, 1024, 65536), _cols(rng, 25600)
        rows = max(1024, min(rows, 300_000_000 // cols))
        shapes = "proj:%dx%d" % (rows, cols)
    elif kind == "attention":
        heads, kv = _log_between(rng, 8, 64) * 128, _log_between(rng, 8, 16) * 128
        shapes = "q_proj:%dx%d k_proj:%dx%d v_proj:%dx%d o_proj:%dx%d" % (heads, hidden, kv, hidden, kv, hidden,
                                                                          max(1024, hidden), heads)
    else:
        inner = max(1024, _log_between(rng, 1024, 25600) // 4 * 4)
        shapes = "gate_proj:%dx%d up_proj:%dx%d down_proj:%dx%d" % (inner, hidden, inner, hidden, hidden, inner)
    c = _linears("", shapes, profile, m, x, rng.random() < 0.4, dist)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs --


def _shapes(case):
    for item in case["shapes"].split():
        name, dims = item.split(":")
        rows, cols = dims.split("x")
        yield name, int(rows), int(cols)


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


def _weight(gen, rows, cols, dist):
    """A bf16 weight on the GPU (made in row slices of bounded size)."""
    w = torch.empty(rows, cols, dtype=torch.bfloat16, device="cuda")
    step = max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        v = _normal(gen, n, cols)
        if dist == "t4":  # unit variance: t4 / sqrt(2), t4 = n / sqrt(chi2_4 / 4)
            chi = sum(_normal(gen, n, cols).square_() for _ in range(4))
            v.div_(chi.div_(4).sqrt_()).mul_(2 ** -0.5)
        w[r:r + n] = v.mul_(0.02)
    return w


def _tensors(case, seed):
    """(name, weight, bias or None) of every Linear of the case, then the
    activations by the first Linear that reads each (q/k/v share one, gate/up
    another): a function of the case and the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shapes = list(_shapes(case)) if case["kind"] == "linears" else [("proj", case["rows"], case["cols"])]
    xs = {}
    for name, _, cols in shapes:
        key = {"k_proj": "q_proj", "v_proj": "q_proj", "up_proj": "gate_proj"}.get(name, name)
        if key not in xs:
            xs[key] = _normal(gen, case.get("m", 1), cols).to(DTYPES[case.get("x", "bf16")])
        xs[name] = xs[key]
    biases = {name: (_normal(gen, rows) * 0.02).to(torch.bfloat16) if case.get("bias") else None
              for name, rows, _ in shapes}
    weights = ((name, _weight(gen, rows, cols, case.get("dist", "normal"))) for name, rows, cols in shapes)
    return weights, biases, xs


def _bits(w):
    return w.view(torch.int16).cpu().numpy().view(np.uint16)


# -------------------------------------------------------------------- cases --


def prepare(case, seed):
    weights, biases, xs = _tensors(case, seed)
    if case["kind"] == "pack":
        # the payload goes into a shard's buffer, as the packer's caller collects it (no tensor
        # that radix compresses outgrows its raw bits)
        shard = np.zeros(case["rows"] * case["cols"] // 2, np.int32)
        return {"kind": "pack", "bits": _bits(next(weights)[1]), "profile": case["profile"], "shard": shard}
    block = torch.nn.Module()
    for name, w in weights:
        if case["kind"] == "narrow":
            lin = torch.nn.Linear(w.shape[1], w.shape[0], bias=biases[name] is not None, device="meta")
            lin.weight = torch.nn.Parameter(w, requires_grad=False)
            if biases[name] is not None:
                lin.bias = torch.nn.Parameter(biases[name], requires_grad=False)
            block.add_module(name, lin)
        else:
            packed = radix_pack.pack_weight_radix(_bits(w), case["profile"])
            block.add_module(name, swap.make_module(packed, biases[name], "cuda"))
    if case["kind"] == "narrow":
        assert swap.install_narrow(block, "cuda")
    else:
        swap.install_groups(block)
    calls = [(module, xs[name]) for name, module in block.named_children()]
    return {"kind": case["kind"], "block": block, "calls": calls}


@torch.no_grad()
def run(state):
    if state["kind"] == "pack":
        p = radix_pack.pack_array_radix(state["bits"], state["profile"])
        state["shard"][:p["rx_data"].size] = p["rx_data"].view(np.int32)
        return [p["rx_palette"], p["rx_offsets"].view(np.int32), state["shard"]]
    return [module(x) for module, x in state["calls"]]


def work(case):
    m = case.get("m", 0)
    size = DTYPES[case.get("x", "bf16")].itemsize
    if case["kind"] == "narrow":
        R, C = case["rows"], case["cols"]
        return {"bytes": 2 * R * C + size * m * (R + C) + (2 * R if case["bias"] else 0), "flops": 2 * m * R * C}
    shapes = list(_shapes(case)) if case["kind"] == "linears" else [("proj", case["rows"], case["cols"])]
    packed = sum(R * C * BITS[case["profile"], case["dist"]] / 8 + 4 * R * -(-C // 1024) for _, R, C in shapes)
    if case["kind"] == "pack":
        return {"bytes": 2 * case["rows"] * case["cols"] + packed, "flops": 0}
    shared = {"k_proj", "v_proj", "up_proj"} if len(shapes) > 1 else set()
    x = sum(m * C * size for name, _, C in shapes if name not in shared)
    out = sum(m * R * size + (2 * R if case["bias"] else 0) for _, R, _ in shapes)
    return {"bytes": packed + x + out, "flops": sum(2 * m * R * C for _, R, C in shapes)}


def tolerance(case):
    """The packed arrays are bytes. Otherwise every weight is exact, sums are
    fp32 and the one rounding is to x's dtype: measured against 64 bits, rel
    is 1.7e-3 (bf16), 2.1e-4 (f16) and 1 to 3e-7 (f32); max is one ulp of the
    output each way."""
    if case["kind"] == "pack":
        return "exact"
    return {"bf16": {"rel": 6e-3, "max": 1.6e-2}, "f16": {"rel": 8e-4, "max": 2e-3},
            "f32": {"rel": 1.2e-6, "max": 1.2e-5}}[case["x"]]


def exact(case, seed):
    if case["kind"] == "pack":
        return None
    weights, biases, xs = _tensors(case, seed)
    out = []
    for name, w in weights:
        x = xs[name].double()
        y = torch.empty(x.shape[0], w.shape[0], dtype=torch.float64, device="cuda")
        step = max(1, (1 << 27) // w.shape[1])
        for r in range(0, w.shape[0], step):
            y[:, r:r + step] = x @ w[r:r + step].double().t()
        out.append(y if biases[name] is None else y + biases[name].double())
    return out
