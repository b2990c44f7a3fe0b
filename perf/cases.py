"""The calls this package is timed on: segmented sum, max and softmax through
``CompiledProgram.run``, as a program that keeps its compiled program and its
output buffer makes them.

A case is one call shape: operation, data type, feature width D, rows N,
segments B, a length distribution, the offsets' type, whether the caller
knows its longest segment (``bound``: passed as ``max_len``), and for a softmax
whether its logits are scaled and masked. Inputs follow from the seed alone:
the lengths are drawn from the distribution and scaled to exactly N rows.
"""
from __future__ import annotations

import atexit
import math
from pathlib import Path
import shutil
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "ragged-mlir_amd"))

from ragged import ArtifactCache, Compiler, ProgramSpec  # noqa: E402

DEVICE = "cuda"
TORCH_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "i32": torch.int32, "i64": torch.int64}
BYTES = {"f32": 4, "bf16": 2, "i32": 4, "i64": 8}
WIDTHS = (1, 2, 3, 4, 5, 8, 16, 25, 32, 46, 64, 84, 100, 128, 168, 256, 500, 1024)
LENGTHS = ("equal", "ragged", "geometric", "exponential", "long_tail", "bimodal", "burst")


def _case(name, op, dtype, d, n, b, lengths, offsets, *, bound=False, scale=1.0, mask=False):
    return {"name": name, "op": op, "dtype": dtype, "d": d, "n": n, "b": b, "lengths": lengths, "offsets": offsets,
            "bound": bound, "scale": scale, "mask": mask}


def listed():
    return [
        # Pooling one small batch of scalar sequences: the call's latency.
        _case("sum_f32_d1_small", "sum", "f32", 1, 32_768, 512, "exponential", "i64"),
        # Softmax over the scores of one small serving batch, 64 columns.
        _case("softmax_bf16_d64_small", "softmax", "bf16", 64, 16_384, 96, "ragged", "i64", bound=True),
        # Ten thousand equal scalar segments (the benchmark's first configuration).
        _case("sum_f32_d1_equal64", "sum", "f32", 1, 640_000, 10_000, "equal", "i64"),
        # Per-neighbourhood attention weights of a large sparse graph: very
        # many very short scalar segments (the benchmark's third configuration).
        _case("softmax_f32_d1_short", "softmax", "f32", 1, 2_790_000, 200_000, "geometric", "i32"),
        # The same operation with a few long runs among single rows (the
        # comparison suite's burst lengths).
        _case("softmax_f32_d1_burst", "softmax", "f32", 1, 1_048_576, 16_384, "burst", "i64", bound=True),
        # Pair features, short segments beside segments of thousands of rows
        # (the benchmark's fourth configuration).
        _case("max_f32_d2_bimodal", "max", "f32", 2, 12_700_000, 50_000, "bimodal", "i32"),
        # Sum pooling of embeddings, segments of up to 512 rows (the
        # benchmark's second configuration).
        _case("sum_f32_d128_ragged512", "sum", "f32", 128, 1_048_576, 4_096, "ragged", "i64"),
        # Max pooling at a width that is no power of two, with padding (-inf)
        # and invalid (NaN) entries among the values.
        _case("max_bf16_d84_exponential", "max", "bf16", 84, 1_000_000, 16_384, "exponential", "i32", bound=True),
        # Sum pooling over a long-tailed corpus: a few segments hold much of the input.
        _case("sum_bf16_d128_long_tail", "sum", "bf16", 128, 4_194_304, 8_192, "long_tail", "i64", bound=True),
        # The comparison suite's long-tail softmax.
        _case("softmax_f32_d128_long_tail", "softmax", "f32", 128, 262_144, 4_096, "long_tail", "i64", bound=True),
        # Attention scores of 16 heads, scaled and with an additive mask.
        _case("softmax_bf16_d16_masked", "softmax", "bf16", 16, 1_000_003, 2_048, "exponential", "i32", bound=True,
              scale=0.125, mask=True),
        # The headline configuration: a 1 GiB long-tail bf16 softmax.
        _case("softmax_bf16_d128_long_tail", "softmax", "bf16", 128, 4_194_304, 8_192, "long_tail", "i64",
              bound=True),
    ]


def draw(rng):
    """A call shape of the same ranges: 64 KiB to 512 MiB of values (a softmax,
    which also writes as much, to 256 MiB), 1 to 200,000 segments."""
    op = rng.choice(("sum", "max", "softmax"))
    dtype = rng.choice(("f32", "bf16"))
    d = rng.choice(WIDTHS)
    most = 28 if op == "softmax" else 29
    n = max(1, int(2 ** rng.uniform(16, most) / (d * BYTES[dtype])))
    b = max(1, int(math.exp(rng.uniform(0, math.log(min(n, 200_000))))))
    masked = op == "softmax" and rng.random() < 0.25
    case = _case("", op, dtype, d, n, b, rng.choice(LENGTHS), rng.choice(("i32", "i64")), bound=rng.random() < 0.5,
                 scale=0.125 if masked else 1.0, mask=masked)
    del case["name"]
    return case


def _offsets(case, seed):
    """[B+1] offsets: segment weights of the distribution, scaled to N rows."""
    rng = np.random.default_rng((seed, 1))
    b, kind = case["b"], case["lengths"]
    if kind == "equal":
        weights = np.ones(b)
    elif kind == "ragged":            # from empty to twice the mean
        weights = rng.uniform(0.0, 2.0, b)
    elif kind == "geometric":
        weights = np.minimum(rng.geometric(1 / 16, b), 32).astype(np.float64)
    elif kind == "exponential":
        weights = rng.exponential(1.0, b)
    elif kind == "long_tail":         # the longest holds about a twentieth of the rows
        weights = rng.pareto(1.2, b) + 1
        weights = np.minimum(weights, max(0.048 * weights.sum(), 1.0))
    elif kind == "bimodal":           # one segment in twenty is about a thousand times longer
        weights = np.where(rng.random(b) < 0.05, rng.uniform(2000, 8000, b), rng.uniform(1, 8, b))
    else:                             # burst: one consecutive hundredth of the segments is long
        weights = np.ones(b)
        width = max(1, b // 100)
        first = int(rng.integers(b - width + 1))
        weights[first:first + width] = 16384
    ends = np.cumsum(weights)
    ends = np.rint(ends * (case["n"] / ends[-1])).astype(np.int64)
    ends[-1] = case["n"]
    return np.concatenate([np.zeros(1, dtype=np.int64), ends])


def _inputs(case, seed):
    """(values, offsets, mask or None, longest segment) on the device."""
    host = _offsets(case, seed)
    n, d = case["n"], case["d"]
    generator = torch.Generator(device=DEVICE).manual_seed(seed * 2 + 1)
    values = torch.randn((n, d), generator=generator, device=DEVICE)
    mask = None
    if case["op"] == "softmax":
        values *= 2.0 if case["scale"] == 1.0 else 16.0     # logits
        if case["mask"]:
            mask = torch.randn((n, d), generator=generator, device=DEVICE)
            mask[torch.rand((n, d), generator=generator, device=DEVICE) < 0.1] = float("-inf")
    elif case["op"] == "max":
        chance = torch.rand((n, d), generator=generator, device=DEVICE)
        values[chance < 1e-4] = float("nan")
        values[chance > 1 - 1e-2] = float("-inf")
    values = values.to(TORCH_DTYPES[case["dtype"]])
    offsets = torch.from_numpy(host).to(DEVICE).to(TORCH_DTYPES[case["offsets"]])
    return values, offsets, mask, int(np.diff(host).max())


_programs = {}
_cache_root = None


def _program(case):
    """The compiled program of the case's specialisation: a program compiles
    it once and keeps it."""
    global _cache_root
    spec = ProgramSpec(case["op"], case["dtype"], case["d"], case["offsets"], scale=case["scale"], mask=case["mask"])
    if spec not in _programs:
        if _cache_root is None:
            _cache_root = tempfile.mkdtemp(prefix="ragged_perf_")
            atexit.register(shutil.rmtree, _cache_root, True)
        _programs[spec] = Compiler().compile(spec, ArtifactCache(_cache_root))
    return _programs[spec]


def prepare(case, seed):
    values, offsets, mask, longest = _inputs(case, seed)
    rows = case["n"] if case["op"] == "softmax" else case["b"]
    out = torch.empty((rows, case["d"]), dtype=values.dtype, device=DEVICE)
    return {"program": _program(case), "values": values, "offsets": offsets, "out": out, "mask": mask,
            "max_len": longest if case["bound"] else None}


def run(state):
    state["program"].run(state["values"], state["offsets"], state["out"], mask=state["mask"], max_len=state["max_len"])
    return state["out"]


def work(case):
    n, b, d, size = case["n"], case["b"], case["d"], BYTES[case["dtype"]]
    rows = n if case["op"] == "softmax" else b
    moved = n * d * size + rows * d * size + (b + 1) * BYTES[case["offsets"]] + (n * d * 4 if case["mask"] else 0)
    # Per element: one add or maximum; a softmax's maximum, subtraction, exponential, sum and division.
    return {"bytes": moved, "flops": n * d * (5 if case["op"] == "softmax" else 1)}


def tolerance(case):
    if case["op"] == "max":
        return "exact"
    # Against float64: bf16 outputs 0.0016-0.0017 (their rounding alone); f32
    # outputs 5e-8 to 8e-8, and sums added one by one in f32 up to 3.4e-7.
    if case["dtype"] == "bf16":
        return {"rel": 7e-3}
    return {"rel": 1.5e-6}


def exact(case, seed):
    values, offsets, mask, _ = _inputs(case, seed)
    offsets = offsets.long()
    x = values.double()
    if case["scale"] != 1.0:
        x = (values.float() * case["scale"]).double()
    if mask is not None:
        x = (x.float() + mask).double()
    if case["op"] == "max":
        return torch.segment_reduce(x, "max", offsets=offsets, axis=0, unsafe=True)
    segments = torch.repeat_interleave(torch.arange(case["b"], device=DEVICE), offsets.diff())
    sums = torch.zeros((case["b"], case["d"]), dtype=torch.float64, device=DEVICE)
    if case["op"] == "sum":
        return sums.index_add_(0, segments, x)
    top = torch.segment_reduce(x, "max", offsets=offsets, axis=0, unsafe=True)
    x = torch.exp(x - top[segments])
    sums.index_add_(0, segments, x)
    return x / sums[segments]
