"""The work that users of this package have it do, as measurable cases through the public entry points.

``grouped_mm`` (forward and training step), its launcher with an fp32 result for weight gradients, and the
mixture-of-experts layer ``moe.moe_forward`` (decode and prefill).  ``listed()`` holds one case per kind of
use, ``draw()`` another one of the same ranges:

    products            2 to 256 groups, 32 to 131072 rows (or columns, or contraction elements) over all groups,
                        K 32 to 14336, N 48 to 14336; bf16, fp16, fp32; group sizes from even to strongly skewed,
                        empty groups among them; second operand row- or column-major; sizes that are not multiples
                        of 8 elements (no aligned vector anywhere) at up to 8e10 FLOP, as fp32
    expert layers       1 to 8192 tokens, 4 to 128 experts, 1 to 8 choices, hidden size 256 to 4096, inner size 128
                        to 14336, weights up to 3 GB; gate and up columns stored apart or interleaved
"""
from __future__ import annotations

import math
import statistics

import torch

from grouped_mm_bf16_amd import grouped_mm, kernels, moe

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
MAX_FLOPS = 2.9e12       # a drawn case costs no more than the largest listed one
MAX_FLOPS_SLOW = 8e10    # fp32 operands and sizes without alignment
MAX_BYTES = 3.0e9


# ---------------------------------------------------------------------------------------------- cases
def _product(variant, G, M, K, N, dtype="bf16", skew=0.4, empty=0, b_col=False, train=False, out_fp32=False):
    """variant 2d3d: M rows in G groups; 3d3d: G products M x K x N; 2d2d: K is split into G groups; 3d2d: N is."""
    return {"op": "product", "variant": variant, "G": G, "M": M, "K": K, "N": N, "dtype": dtype, "skew": skew,
            "empty": empty, "b_col": b_col, "train": train, "out_fp32": out_fp32}


def _layer(tokens, experts, top_k, hidden, inner, interleaved, skew=0.5, dtype="bf16", logits="fp32"):
    return {"op": "layer", "T": tokens, "E": experts, "top_k": top_k, "H": hidden, "I": inner,
            "interleaved": interleaved, "skew": skew, "dtype": dtype, "logits": logits}


def listed():
    cases = {
        # the first thing a user tries: the README's call, a handful of rows in six groups, two of them empty
        "readme": _product("2d3d", 6, 32, 64, 48, empty=2),
        # the benchmark program's default sizes, forward and backward: many rows, very narrow matrices
        "narrow_train": _product("2d3d", 64, 131072, 32, 64, skew=0.0, train=True),
        # one decoding step of a served model with few large experts: 32 sequences
        "decode_large_experts": _layer(32, 8, 2, 4096, 14336, interleaved=False),
        # one decoding step of a served model with many small experts: 64 sequences
        "decode_small_experts": _layer(64, 128, 8, 2048, 768, interleaved=True),
        # a prompt batch through the large experts, weights prepared for the fused activation
        "prefill_large_experts": _layer(8192, 8, 2, 4096, 14336, interleaved=True),
        # a prompt batch through the small experts, weights as published (gate and up columns apart)
        "prefill_small_experts": _layer(4096, 128, 8, 2048, 768, interleaved=False, skew=1.0),
        # the up projection alone, as a user's own layer code calls it: the headline product
        "up_projection": _product("2d3d", 8, 16384, 4096, 14336),
        # training step of a fine-grained expert layer, weights stored as linear layers store them
        "train_small_experts": _product("2d3d", 128, 32768, 2048, 768, skew=2.4, empty=20, b_col=True, train=True),
        # a batch of equal products (per-head or per-expert with fixed capacity), half precision
        "batched": _product("3d3d", 32, 1024, 1024, 4096, dtype="fp16"),
        # accumulating weight gradients in fp32: the contraction (tokens) is what the groups split
        "weight_grad_fp32": _product("2d2d", 8, 4096, 16384, 14336, out_fp32=True),
        # full precision, columns split over the groups
        "columns_fp32": _product("3d2d", 8, 1024, 1024, 8192, dtype="fp32"),
        # a training step whose sizes have no alignment at all
        "odd_train": _product("2d3d", 24, 6151, 1031, 519, skew=1.0, empty=2, train=True),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log(rng, lo, hi):
    """Whole number between lo and hi, uniform in its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _draw_product(rng):
    variant = rng.choice(["2d3d", "2d3d", "2d3d", "3d3d", "2d2d", "3d2d"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    odd = rng.random() < 0.25
    train = variant in ("2d3d", "3d3d") and rng.random() < 0.4
    G = _log(rng, 2, 256 if variant == "2d3d" else 48)
    jagged = _log(rng, 32, 131072 if variant == "2d3d" else 16384)
    M, K, N = _log(rng, 64, 4096), _log(rng, 32, 14336), _log(rng, 48, 14336)
    if variant == "2d3d":
        M = jagged
    elif variant == "2d2d":
        K = jagged
    elif variant == "3d2d":
        N = jagged
    if not odd:
        M, K, N = (max(8, x // 8 * 8) for x in (M, K, N))
        if variant == "2d3d":
            M += rng.randrange(8)      # rows are contiguous along K: their number needs no alignment
    case = _product(variant, G, M, K, N, dtype=dtype, skew=rng.choice([0.0, 0.4, 1.0, 2.4]),
                    empty=rng.choice([0, 0, G // 8, G // 3]), b_col=rng.random() < 0.5, train=train,
                    out_fp32=variant == "2d2d" and dtype != "fp32" and rng.random() < 0.5)
    return case, odd or dtype == "fp32"


def draw(rng):
    while True:
        if rng.random() < 0.35:
            hidden, inner = 8 * _log(rng, 32, 512), 64 * _log(rng, 2, 224)
            experts = _log(rng, 4, 128)
            case = _layer(_log(rng, 1, 8192), experts, rng.randint(1, min(8, experts)), hidden, inner,
                          interleaved=rng.random() < 0.5, skew=rng.choice([0.0, 0.5, 1.0]),
                          dtype=rng.choice(["bf16", "bf16", "fp16"]), logits=rng.choice(["fp32", "bf16"]))
            slow = False
            weights = 3 * experts * hidden * inner * 2
        else:
            case, slow = _draw_product(rng)
            weights = 0
        need = work(case)
        if need["flops"] <= (MAX_FLOPS_SLOW if slow else MAX_FLOPS) and max(need["bytes"], weights) <= MAX_BYTES:
            return case


# ---------------------------------------------------------------------------------------------- inputs
def _group_sizes(total, groups, skew, empty, seed):
    """Sizes of `groups` groups that sum to `total`.  `empty` of them are empty, the others hold at least one
    element and follow a saturating log-normal profile (no expert gets every token); the seed shuffles which
    group is which and moves a few elements between them."""
    used = max(1, min(groups - empty, total))
    normal = statistics.NormalDist()
    shares = [1.0 / (math.exp(-skew * normal.inv_cdf((i + 0.5) / used)) + 0.01) for i in range(used)]
    rest, whole = total - used, sum(shares)
    sizes = [1 + int(rest * s / whole) for s in shares]
    sizes[-1] += total - sum(sizes)
    gen = torch.Generator().manual_seed(seed)
    if skew:
        pairs = torch.randint(0, used, (used, 2), generator=gen).tolist()
        parts = torch.rand(used, generator=gen).tolist()
        for (i, j), part in zip(pairs, parts):
            moved = int(0.1 * part * (sizes[i] - 1))
            sizes[i] -= moved
            sizes[j] += moved
    sizes += [0] * (groups - used)
    order = torch.randperm(groups, generator=gen).tolist()
    return [sizes[i] for i in order]


def _random(gen, shape, dtype, scale=1.0):
    t = torch.randn(shape, device=DEVICE, dtype=dtype, generator=gen)
    return t if scale == 1.0 else t.mul_(scale)


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    if case["op"] == "layer":
        T, E, H, inner = case["T"], case["E"], case["H"], case["I"]
        popularity = case["skew"] * torch.randn(E, device=DEVICE, generator=gen)
        logits = torch.randn(T, E, device=DEVICE, generator=gen) + popularity
        w_up = _random(gen, (E, H, 2 * inner), dtype, 0.02)
        if case["interleaved"]:
            w_up = moe.interleave_gate_up(w_up)
        return {"op": "layer", "x": _random(gen, (T, H), dtype), "logits": logits.to(DTYPES[case["logits"]]),
                "w_up": w_up, "w_down": _random(gen, (E, inner, H), dtype, 0.02), "top_k": case["top_k"],
                "interleaved": case["interleaved"]}
    G, M, K, N, variant = case["G"], case["M"], case["K"], case["N"], case["variant"]
    a_shape = {"2d3d": (M, K), "3d3d": (G, M, K), "2d2d": (M, K), "3d2d": (G, M, K)}[variant]
    b_shape = {"2d3d": (G, K, N), "3d3d": (G, K, N), "2d2d": (K, N), "3d2d": (K, N)}[variant]
    out_shape = {"2d3d": (M, N), "3d3d": (G, M, N), "2d2d": (G, M, N), "3d2d": (M, N)}[variant]
    a = _random(gen, a_shape, dtype)
    scale = 1.0 if variant == "2d2d" else 0.02     # activations and their gradients; otherwise weights
    if case["b_col"]:
        b = _random(gen, b_shape[:-2] + (b_shape[-1], b_shape[-2]), dtype, scale).transpose(-2, -1)
    else:
        b = _random(gen, b_shape, dtype, scale)
    offs = None
    if variant != "3d3d":
        sizes = _group_sizes({"2d3d": M, "2d2d": K, "3d2d": N}[variant], G, case["skew"], case["empty"], seed)
        offs = torch.tensor(sizes, dtype=torch.int64).cumsum(0).to(torch.int32).to(DEVICE)
    state = {"op": "product", "a": a, "b": b, "offs": offs, "train": case["train"]}
    if case["train"]:
        a.requires_grad_()
        b.requires_grad_()
        state["grad_out"] = _random(gen, out_shape, dtype)
    if case["out_fp32"]:
        state["out"] = torch.zeros(out_shape, device=DEVICE, dtype=torch.float32)   # a gradient buffer a trainer keeps
    return state


# ---------------------------------------------------------------------------------------------- one pass
def run(state):
    if state["op"] == "layer":
        return moe.moe_forward(state["x"], state["logits"], state["w_up"], state["w_down"], state["top_k"],
                               interleaved=state["interleaved"])
    a, b, offs = state["a"], state["b"], state["offs"]
    if "out" in state:
        kernels.grouped_mm_2d2d(a, b, offs, state["out"])
        return state["out"]
    out = grouped_mm(a, b, offs=offs)
    if not state["train"]:
        return out
    grad_a, grad_b = torch.autograd.grad(out, (a, b), state["grad_out"])
    return {"out": out.detach(), "grad_a": grad_a, "grad_b": grad_b}


# ---------------------------------------------------------------------------------------------- what it takes
def work(case):
    size = BYTES[case["dtype"]]
    if case["op"] == "layer":
        T, E, k, H, inner = case["T"], case["E"], case["top_k"], case["H"], case["I"]
        touched = E * (1.0 - (1.0 - k / E) ** T)      # experts that at least one token chooses
        per_expert = 3 * H * inner
        return {"bytes": int(size * (2 * T * H + touched * per_expert) + T * E * BYTES[case["logits"]]),
                "flops": 2 * T * k * per_expert}
    G, M, K, N, variant = case["G"], case["M"], case["K"], case["N"], case["variant"]
    total = {"2d3d": M, "3d3d": G, "2d2d": K, "3d2d": N}[variant]
    used = G if variant == "3d3d" else max(1, min(G - case["empty"], total))
    a = {"2d3d": M * K, "3d3d": G * M * K, "2d2d": M * K, "3d2d": used * M * K}[variant]
    b = {"2d3d": used * K * N, "3d3d": G * K * N, "2d2d": K * N, "3d2d": K * N}[variant]
    out = {"2d3d": M * N, "3d3d": G * M * N, "2d2d": G * M * N, "3d2d": M * N}[variant]
    flops = 2 * M * K * N * (G if variant == "3d3d" else 1)
    moved = (a + b) * size + out * (4 if case["out_fp32"] else size)
    if case["train"]:
        # backward: the output's gradient in, both operands' gradients out (every group's, the empty ones' too)
        moved += (out + a + (G * K * N if variant == "2d3d" else b)) * size
        flops *= 3
    return {"bytes": int(moved), "flops": int(flops)}


def tolerance(case):
    """Four times the difference from the same path in 64 bits, as measured on the listed cases: the rounding of the
    result (and of the layer's two intermediates) to its type (bf16 product 1.66e-3, largest 3.9e-3 of the value;
    layer 3.9e-3, largest 2.3e-2; fp16 an eighth of that), or the error of an fp32 sum (5.7e-7, largest 5.4e-6 at
    1024 terms; it grows like the square root of their number)."""
    if case["dtype"] == "fp32" or case.get("out_fp32"):
        terms = max(case["K"], case["M"] // 4 if case["train"] else 0)
        grow = max(1.0, math.sqrt(terms / 1024))
        return {"rel": 2.3e-6 * grow, "max": 2.2e-5 * grow}
    unit = 1.0 if case["dtype"] == "bf16" else 0.125
    if case["op"] == "layer":
        return {"rel": 1.55e-2 * unit, "max": 9e-2 * unit}
    return {"rel": 6.6e-3 * unit, "max": 1.6e-2 * unit}
