"""Measured cases of the expert-GEMM path, through the package's public entry points.

Each case is a dict of plain values.  ``kind`` names the call a program makes:

* ``group``    ``launch_grouped`` over G equal problems (one rank's experts, packed W13 or W2);
* ``ragged``   ``launch_grouped`` over per-expert tensors of unequal row counts (a router's result
               held as one tensor per expert);
* ``routed``   ``grouped_mm`` over expert-sorted rows with device offsets;
* ``swiglu``   ``grouped_mm_swiglu`` over expert-sorted rows (packed Gate+Up with the activation);
* ``gate_up``  ``launch_gate_up_swiglu`` over G equal problems;
* ``linear``   ``launch_matmul`` with a weight stored [N, K] as linear layers store it (B is its
               transposed view);
* ``backward`` the two products of a GEMM's backward pass, dA = dC B^T and dB = A^T dC, as two
               ``launch_matmul`` calls on transposed views;
* ``matmul``   ``launch_matmul`` on row-major operands.

Calls whose shapes repeat use the launchers as they are (the first call of a shape measures the
candidates and later calls look the result up).  Calls whose row counts follow the router differ
from step to step, so a serving program passes ``autotune=False`` there; those cases do the same.
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PACKAGE = os.path.join(_ROOT, "moe-gemm-parallel-bench_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from kernels import grouped_mm, grouped_mm_swiglu, launch_gate_up_swiglu, launch_grouped, launch_matmul  # noqa: E402
from kernels.grouped_gemm import workspace_from_tensors  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}
_ROUTED = ("ragged", "routed", "swiglu")  # M is the mean row count of an expert


def _case(kind, g, m, k, n, dtype="bf16", precision="ieee", **more):
    return dict(kind=kind, G=g, M=m, K=k, N=n, dtype=dtype, precision=precision, **more)


def listed():
    return [
        # The smallest group of the test configurations: 8 experts, 64 tokens each.  Launch latency.
        _case("group", 8, 64, 512, 1024, name="group_small"),
        # Packed W13 of one of 8 expert-parallel ranks (32 experts), decode: 8 tokens an expert.
        # Reads 1.9 GB of weights.
        _case("group", 32, 8, 7168, 4096, name="w13_decode"),
        # The same rank in prefill, 512 tokens an expert: the benchmark's headline and the largest case.
        _case("group", 32, 512, 7168, 4096, name="w13_prefill"),
        # Tensor-parallel shard of a small-expert model (N = 2 x 192 columns), 128 experts, fp16.
        _case("group", 128, 32, 2048, 384, "fp16", name="tp_w13_fp16"),
        # Expert-sorted prefill batch, 2048 tokens x top-4 over 128 experts, sizes that are no
        # multiple of a tile (2880); row counts from the router.
        _case("routed", 128, 64, 2880, 5760, name="routed_prefill"),
        # Fused Gate+Up of a decode step: 64 tokens x top-8 over 128 experts, most experts hold a few rows.
        _case("swiglu", 128, 4, 2048, 1536, name="routed_swiglu_decode"),
        # W2 over per-expert tensors of unequal row counts (one rank's 32 experts, chunked prefill).
        _case("ragged", 32, 200, 2048, 7168, name="ragged_w2"),
        # A linear layer's weight [N, K] at 16 tokens (decode of a dense or shared expert).
        _case("linear", 1, 16, 4096, 14336, name="linear_decode"),
        # Backward of an expert's W13 shard at 1024 tokens.
        _case("backward", 1, 1024, 4096, 3584, name="backward"),
        # Odd extents: no row is 16-byte aligned.
        _case("matmul", 1, 777, 2881, 1443, "fp16", name="odd_fp16"),
        # fp32 experts (the default input precision), 8 experts.
        _case("group", 8, 512, 2048, 1536, "fp32", name="group_fp32"),
        # fp32 operands at TF32 input precision, one expert (a G = 1 group is a single GEMM).
        _case("group", 1, 1024, 4096, 3584, "fp32", "tf32", name="expert_tf32"),
    ]


# Most FLOP of a drawn case by the way it runs: no drawn case takes longer than the largest listed one.
_FLOP_CAP = 2.0e11
_FLOP_CAP_SLOW = 2.0e10  # fp32, transposed and unaligned operands
_WEIGHT_CAP = 1.0e9      # weight bytes


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kinds = ("group", "group", "group", "ragged", "routed", "swiglu", "gate_up", "linear", "backward", "matmul")
    while True:
        kind = rng.choice(kinds)
        dtype = rng.choice(("bf16", "bf16", "fp16"))
        precision = "ieee"
        if kind in ("group", "matmul") and rng.random() < 0.35:
            dtype, precision = "fp32", rng.choice(("ieee", "tf32"))
        g = 1 if kind in ("linear", "backward", "matmul") else _log_uniform(rng, 2, 128)
        if kind == "gate_up":
            g = min(g, 32)
        k, n = _log_uniform(rng, 256, 7168), _log_uniform(rng, 256, 7168)
        if kind == "matmul":  # any extents, odd ones among them
            m = _log_uniform(rng, 1, 2048)
        else:  # model widths are multiples of 16
            k, n = max(256, k // 16 * 16), max(256, n // 16 * 16)
            m = _log_uniform(rng, 64, 2048) if kind == "backward" else _log_uniform(rng, 1, 1024)
        case = _case(kind, g, m, k, n, dtype, precision)
        slow = dtype == "fp32" or kind in ("linear", "backward", "matmul")
        if work(case)["flops"] <= (_FLOP_CAP_SLOW if slow else _FLOP_CAP) and g * k * n * _SIZES[dtype] <= _WEIGHT_CAP:
            return case


def _row_counts(case, generator):
    """Rows of each expert: G x M rows routed by uneven expert popularity (some experts get none)."""
    g = case["G"]
    popularity = torch.randn(g, generator=generator).mul_(0.6).exp_()
    choice = torch.multinomial(popularity, g * case["M"], replacement=True, generator=generator)
    return torch.bincount(choice, minlength=g).tolist()


def _operands(case, seed):
    """Activations ~ N(0, 1), weights ~ N(0, 0.02) (gradients ~ N(0, 0.02)), drawn on the GPU."""
    generator = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal(shape, scale):
        return torch.empty(shape, device="cuda", dtype=dtype).normal_(generator=generator).mul_(scale)

    g, m, k, n, kind = (case[f] for f in ("G", "M", "K", "N", "kind"))
    if kind in _ROUTED:
        return {"a": normal((g * m, k), 1.0), "b": normal((g, k, n), 0.02),
                "rows": _row_counts(case, torch.Generator().manual_seed(seed))}
    if kind in ("group", "gate_up"):
        return {"a": normal((g, m, k), 1.0), "b": normal((g, k, n), 0.02)}
    if kind == "linear":
        return {"a": normal((m, k), 1.0), "w": normal((n, k), 0.02)}
    if kind == "backward":
        return {"a": normal((m, k), 1.0), "b": normal((k, n), 0.02), "dc": normal((m, n), 0.02)}
    return {"a": normal((m, k), 1.0), "b": normal((k, n), 0.02)}


def _expert_rows(rows):
    """(expert, first row, end row) of the experts that hold rows."""
    first = 0
    for e, count in enumerate(rows):
        if count:
            yield e, first, first + count
        first += count


def prepare(case, seed):
    x = _operands(case, seed)
    kind, m, n = case["kind"], case["M"], case["N"]
    state = {"kind": kind, "precision": case["precision"], **x}
    like = x["a"]
    if kind in ("group", "gate_up"):
        state["c"] = like.new_empty((case["G"], m, n))
        state["workspace"] = workspace_from_tensors(list(x["a"]), list(x["b"]), list(state["c"]))
    elif kind == "ragged":
        state["c"] = like.new_empty((case["G"] * m, n))
        spans = list(_expert_rows(x["rows"]))
        state["workspace"] = workspace_from_tensors([x["a"][r0:r1] for _, r0, r1 in spans],
                                                    [x["b"][e] for e, _, _ in spans],
                                                    [state["c"][r0:r1] for _, r0, r1 in spans])
    elif kind in ("routed", "swiglu"):
        state["offs"] = torch.tensor(x["rows"], device="cuda").cumsum(0).to(torch.int32)
        state["c"] = like.new_empty((case["G"] * m, n if kind == "routed" else n // 2))
    elif kind == "backward":
        state["da"], state["db"] = torch.empty_like(x["a"]), torch.empty_like(x["b"])
    else:
        state["c"] = like.new_empty((m, n))
    return state


def run(state):
    kind = state["kind"]
    if kind == "group":
        launch_grouped(state["workspace"], state["precision"])
        return state["c"]
    if kind == "gate_up":
        return launch_gate_up_swiglu(state["workspace"])
    if kind == "ragged":
        launch_grouped(state["workspace"], autotune=False)
        return state["c"]
    if kind == "routed":
        return grouped_mm(state["a"], state["b"], state["offs"], out=state["c"], autotune=False)
    if kind == "swiglu":
        return grouped_mm_swiglu(state["a"], state["b"], state["offs"], out=state["c"], autotune=False)
    if kind == "linear":
        launch_matmul(state["a"], state["w"].t(), state["c"])
        return state["c"]
    if kind == "backward":
        launch_matmul(state["dc"], state["b"].t(), state["da"])
        launch_matmul(state["a"].t(), state["dc"], state["db"])
        return {"da": state["da"], "db": state["db"]}
    launch_matmul(state["a"], state["b"], state["c"], input_precision=state["precision"])
    return state["c"]


def work(case):
    g, m, k, n = (case[f] for f in ("G", "M", "K", "N"))
    products = 2 if case["kind"] == "backward" else 1
    out = n // 2 if case["kind"] in ("swiglu", "gate_up") else n
    values = g * (m * k + k * n + m * out)
    if case["kind"] == "backward":  # reads dC, B and A once, writes dA and dB
        values = m * n + 2 * k * n + 2 * m * k
    return {"bytes": float(values * _SIZES[case["dtype"]]), "flops": 2.0 * products * g * m * k * n}


def tolerance(case):
    # About four times the measured error against 64 bits.  Rounding of the output dominates in 16
    # bits (1.7e-3 in bf16, 2.1e-4 in fp16); fp32 results differ by the order of their sums
    # (0.8e-6 to 1.1e-6 at K = 2048 to 4096, growing with K).
    if case["dtype"] == "fp32":
        return {"rel": 6e-6, "max": 2e-4}
    return {"rel": 7e-3, "max": 0.04} if case["dtype"] == "bf16" else {"rel": 9e-4, "max": 5e-3}


def _tf32(x):
    """fp32 values rounded to TF32's 10-bit mantissa, ties away from zero."""
    bits = x.view(torch.int32)
    return ((bits + 0x1000) & -0x2000).view(torch.float32)


def exact(case, seed):
    x = _operands(case, seed)
    kind = case["kind"]

    def mm(a, b):
        if case["precision"] == "tf32":
            a, b = _tf32(a), _tf32(b)
        return torch.mm(a.double(), b.double())

    def swiglu(y):
        gate, up = y.chunk(2, dim=1)
        return torch.nn.functional.silu(gate) * up

    if kind == "gate_up":
        return [swiglu(mm(a, b)) for a, b in zip(x["a"], x["b"])]
    if kind == "group":
        return torch.stack([mm(a, b) for a, b in zip(x["a"], x["b"])])
    if kind in _ROUTED:
        parts = [mm(x["a"][r0:r1], x["b"][e]) for e, r0, r1 in _expert_rows(x["rows"])]
        return torch.cat([swiglu(p) for p in parts] if kind == "swiglu" else parts)
    if kind == "linear":
        return mm(x["a"], x["w"].t())
    if kind == "backward":
        return {"da": mm(x["dc"], x["b"].t()), "db": mm(x["a"].t(), x["dc"])}
    return mm(x["a"], x["b"])
