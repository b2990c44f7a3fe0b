"""The tile schedule of sum and max (csrc/tiles.hpp) against the oracle, at the
sizes where it can go wrong: one tile, one workgroup of tiles, many tiles;
segments inside a batch of a wave (several at once from LDS, and longer ones
among them), across batches, across tiles and over more tiles than one lane
folds; empty segments at both ends and between; array ends inside a vector;
every access width, the flat mapping and the widest rows (64 lanes)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ragged import runtime
from ragged import Compiler, Optimizations, ProgramSpec
from ragged.workloads import offsets_from_lengths

pytestmark = pytest.mark.gpu

GEOMETRIES = [("f32", 1), ("f32", 2), ("f32", 3), ("f32", 4), ("f32", 6), ("f32", 16), ("f32", 25), ("f32", 128),
              ("f32", 256), ("bf16", 1), ("bf16", 2), ("bf16", 4), ("bf16", 5), ("bf16", 8),
              ("bf16", 84), ("bf16", 128), ("bf16", 512)]


def lengths_of(kind, d, elements):
    """Lengths of about ``elements`` values in all."""
    rng = np.random.default_rng(len(kind) * 1000 + d)
    rows = max(6, elements // d)
    if kind == "tiny":              # zero to three rows, empty runs at both ends
        lengths = rng.integers(0, 4, max(8, rows // 2))
        lengths[:5] = lengths[-70:] = 0
    elif kind == "middle":          # around a batch of a wave
        lengths = rng.integers(1, max(2, 2 * (1024 // d) + 3), max(3, rows // (1024 // d + 2)))
    elif kind == "spread":          # one long segment in sixteen among short ones
        lengths = np.where(np.arange(max(8, rows // 40)) % 16 == 7, 600 // min(d, 32) + 17, rng.integers(1, 6))
    else:                           # one segment holds nearly everything
        lengths = np.array([3, 0, rows + 1, 1, 0])
    return lengths.astype(np.int64)


@pytest.mark.parametrize("dtype,d", GEOMETRIES)
@pytest.mark.parametrize("op", ["sum", "max"])
def test_tiles_match_the_oracle(artifact_cache, monkeypatch, op, dtype, d):
    from gpu_helpers import check, run_program
    offsets_dtype = "i32" if d % 2 else "i64"
    program = Compiler().compile(ProgramSpec(op, dtype, d, offsets_dtype), artifact_cache)
    launches = set()
    monkeypatch.setattr(runtime, "SMALL_SEGMENTS", 0)      # small calls too
    monkeypatch.setattr(runtime, "CLASSIFIED_LANES", 0)    # and many short segments
    for elements in (700, 40_000, 900_000):
        for kind in ("tiny", "middle", "spread", "one"):
            offsets = offsets_from_lengths(lengths_of(kind, d, elements), offsets_dtype)
            values = np.random.default_rng(7).normal(size=(int(offsets[-1]), d)).astype(np.float32)
            print(op, dtype, d, kind, values.shape, len(offsets) - 1, flush=True)
            actual, report = run_program(program, values, offsets, dtype=dtype, op=op)
            assert report.selection.get("tiles") and report.kernel_names[0].endswith("split_partial")
            launches.add(len(report.kernel_names))
            check(actual, values, offsets, op=op, dtype=dtype)
    assert launches == {1, 2}       # one workgroup, and tiles folded by a second launch


@pytest.mark.parametrize("op,dtype,d", [("sum", "f32", 1), ("max", "bf16", 5), ("sum", "bf16", 16)])
def test_tiles_element_access(artifact_cache, op, dtype, d):
    """One element per access, non-finite values."""
    from gpu_helpers import check, run_program
    program = Compiler().compile(ProgramSpec(op, dtype, d, "i64", optimizations=Optimizations(vectorize=False)),
                                 artifact_cache)
    rng = np.random.default_rng(3)
    offsets = offsets_from_lengths(rng.integers(0, 90, 900).astype(np.int64), "i64")
    values = rng.normal(size=(int(offsets[-1]), d)).astype(np.float32)
    values[rng.random(values.shape) < 0.003] = np.nan
    values[rng.random(values.shape) < 0.003] = -np.inf
    actual, report = run_program(program, values, offsets, dtype=dtype, op=op)
    assert report.selection.get("tiles")
    check(actual, values, offsets, op=op, dtype=dtype)


@pytest.mark.parametrize("op", ["sum", "max"])
@pytest.mark.parametrize("dtype,d,vectorize", [("f32", 2, True), ("bf16", 2, True), ("bf16", 4, True), ("f32", 2, False),
                                               ("f32", 6, False), ("bf16", 1, False), ("bf16", 4, False), ("bf16", 60, False)])
def test_tiles_on_views_at_any_element(artifact_cache, monkeypatch, op, dtype, d, vectorize):
    """Results of a flat-mapped program at any element of a buffer (its values
    are aligned), and values and results of one with element accesses."""
    from gpu_helpers import check, torch_dtype
    monkeypatch.setattr(runtime, "SMALL_SEGMENTS", 0)
    program = Compiler().compile(ProgramSpec(op, dtype, d, "i64", optimizations=Optimizations(vectorize=vectorize)),
                                 artifact_cache)
    rng = np.random.default_rng(d)
    for lengths in (rng.integers(0, 90, 900), [5, 0, 9000, 3], [3]):
        offsets = offsets_from_lengths(np.array(lengths, dtype=np.int64), "i64")
        n, b = int(offsets[-1]), len(offsets) - 1
        values = rng.normal(size=(n, d)).astype(np.float32)
        for shift in (1, 3):
            x = torch.zeros(n * d + 16, dtype=torch_dtype(torch, dtype), device="cuda")
            y = torch.full((b * d + 16,), -64.0, dtype=x.dtype, device="cuda")
            first = 0 if vectorize else shift
            x[first:first + n * d] = torch.from_numpy(values).reshape(-1).to("cuda")
            out = y[shift:shift + b * d].view(b, d)
            report = program.run(x[first:first + n * d].view(n, d), torch.from_numpy(offsets).to("cuda"), out)
            assert report.selection.get("tiles")
            check(out.float().cpu().numpy().astype(np.float64), values, offsets, op=op, dtype=dtype)
            assert bool((y[:shift] == -64).all()) and bool((y[shift + b * d:] == -64).all())


@pytest.mark.parametrize("d", [4, 64, 84, 128])
def test_tiles_bf16_sums_of_infinities(artifact_cache, d):
    """Rows added several at a time and again one by one where a sum is not
    finite: short segments with infinities of one sign, of both, and NaN,
    among finite columns."""
    from gpu_helpers import check, run_program
    program = Compiler().compile(ProgramSpec("sum", "bf16", d, "i64"), artifact_cache)
    rng = np.random.default_rng(d)
    lengths = np.concatenate([rng.integers(1, 200, 300), [60_000 // d]]).astype(np.int64)
    offsets = offsets_from_lengths(lengths, "i64")
    values = rng.normal(size=(int(offsets[-1]), d)).astype(np.float32)
    values[rng.random(values.shape) < 0.004] = np.inf
    values[:len(values) // 2][rng.random((len(values) // 2, d)) < 0.002] = -np.inf
    values[rng.random(values.shape) < 0.001] = np.nan
    actual, report = run_program(program, values, offsets, dtype="bf16", op="sum")
    assert report.selection.get("tiles")
    check(actual, values, offsets, op="sum", dtype="bf16")


def extremes(n, d, rng):
    """Finite values but for column 0 (one +inf) and, in rows of four or more, 1
    (one -inf), 2 (both) and 3 (two finite values whose sum overflows); no NaN."""
    values = rng.normal(size=(n, d)).astype(np.float32)
    near, far = n // 5, n - n // 7
    values[far, 0] = np.inf
    if d > 3:
        values[near, 1] = -np.inf
        values[near, 2], values[far, 2] = np.inf, -np.inf
        values[near, 3] = values[far, 3] = 3e38
    return values


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("d,parts", [(1, 8), (1, 24), (1, 60), (1, 1000), (4, 24), (4, 60), (4, 900), (4, 1500), (64, 24),
                                     (64, 60), (64, 200), (64, 900), (84, 100), (128, 600)])
def test_tiles_infinite_sums_of_long_segments(artifact_cache, monkeypatch, dtype, d, parts):
    """A sum that is infinite, or overflows, is infinite however many tiles
    its segment crosses: chains a lane folds (up to 32 parts), a wave (64 per
    lane group) and a workgroup, and those of a single workgroup of tiles."""
    from gpu_helpers import run_program
    monkeypatch.setattr(runtime, "SMALL_SEGMENTS", 0)
    program = Compiler().compile(ProgramSpec("sum", dtype, d, "i64"), artifact_cache)
    row = d * (2 if dtype == "bf16" else 4)
    n = parts * (1 << 10 if parts <= 1000 else 4 << 10) // row
    rng = np.random.default_rng(parts)
    values = np.concatenate([rng.normal(size=(2, d)).astype(np.float32), extremes(n, d, rng),
                             rng.normal(size=(3, d)).astype(np.float32)])
    offsets = np.array([0, 2, n + 2, n + 5], dtype=np.int64)
    for flip in (1, -1):
        actual, report = run_program(program, values * np.float32(flip), offsets, dtype=dtype, op="sum")
        assert report.selection.get("tiles")
        assert np.isfinite(actual[[0, 2]]).all()
        assert actual[1, 0] == flip * np.inf
        if d > 3:
            assert actual[1, 1] == -flip * np.inf and np.isnan(actual[1, 2]) and actual[1, 3] == flip * np.inf
            assert np.isfinite(actual[1, 4:]).all()


@pytest.mark.parametrize("op,dtype,d", [("sum", "f32", 2), ("sum", "bf16", 128), ("max", "f32", 100)])
def test_tiles_repeat_bit_for_bit_and_share_a_workspace(artifact_cache, op, dtype, d):
    """The chains' order does not depend on scheduling, and a call on the
    classified schedule between (same workspace) changes nothing."""
    from gpu_helpers import run_program
    program = Compiler().compile(ProgramSpec(op, dtype, d, "i64"), artifact_cache)
    rng = np.random.default_rng(11)
    lengths = np.concatenate([[300_000 // d], rng.integers(0, 300, 2000)]).astype(np.int64)
    offsets = offsets_from_lengths(lengths, "i64")
    values = rng.normal(size=(int(offsets[-1]), d)).astype(np.float32)
    first, _ = run_program(program, values, offsets, dtype=dtype, op=op)
    classified, _ = run_program(program, values, offsets, dtype=dtype, op=op, select="classified")
    again, _ = run_program(program, values, offsets, dtype=dtype, op=op)
    classified_again, _ = run_program(program, values, offsets, dtype=dtype, op=op, select="classified")
    assert np.array_equal(first, again) and np.array_equal(classified, classified_again)


@pytest.mark.parametrize("op,dtype,d", [("sum", "f32", 1), ("max", "bf16", 5)])
def test_small_calls_run_block_per_segment(artifact_cache, monkeypatch, op, dtype, d):
    """A call that fits the small rule is one launch; one segment more, one
    row more or an unknown longest segment beyond it is not (larger calls'
    estimates aside)."""
    monkeypatch.setattr(runtime.ReduceEstimate, "blocks", lambda *_: float("inf"))
    from gpu_helpers import check, run_program
    program = Compiler().compile(ProgramSpec(op, dtype, d, "i32"), artifact_cache)
    row = d * (2 if dtype == "bf16" else 4)
    most = runtime.SMALL_LONGEST_PER_ACCESS * (16 if d == 1 else 2) // row       # rows of the longest segment
    rng = np.random.default_rng(2)
    for lengths, max_len, small in (([most, 0, 3], most, True), ([most, 0, 3], None, False), ([most - 3, 0, 3], None, True),
                                    ([most + 1, 5], most + 1, False), ([2] * runtime.SMALL_SEGMENTS, 2, True),
                                    ([70] * (runtime.SMALL_SEGMENTS + 1), 70, False)):
        offsets = offsets_from_lengths(np.array(lengths, dtype=np.int64), "i32")
        values = rng.normal(size=(int(offsets[-1]), d)).astype(np.float32)
        actual, report = run_program(program, values, offsets, dtype=dtype, op=op, max_len=max_len)
        assert report.selected == ("naive" if small else "classified")
        assert bool(report.selection.get("tiles")) != small
        check(actual, values, offsets, op=op, dtype=dtype)


@pytest.mark.parametrize("op,dtype,d,lengths,max_len,route", [
    # every segment reduced alone by a lane group (a small call: block per segment)
    ("sum", "f32", 16, [32] * 5000, 32, "alone"), ("max", "bf16", 128, [7, 0, 32] * 3000, 32, "alone"),
    ("sum", "f32", 16, [32] * 4096, 32, "naive"), ("sum", "f32", 16, [33] * 12_000, 33, "tiles"),
    # many segments of some hundred rows, and with one that one workgroup would take long for
    ("max", "f32", 3, [500] * 7600, 500, "naive"), ("max", "f32", 3, [500] * 7600 + [40_000], 40_000, "tiles"),
    ("max", "f32", 3, [500] * 7600, None, "tiles"), ("sum", "bf16", 46, [80] * 7600, 80, "naive"),
    # many short segments of unknown length: narrow rows, wide rows, fewer, longer
    ("sum", "f32", 16, [10] * 5000, None, "classified"), ("sum", "f32", 128, [10] * 5000, None, "tiles"),
    ("sum", "f32", 16, [10] * 4999, None, "tiles"), ("sum", "f32", 16, [16] * 5000, None, "tiles"),
    ("sum", "f32", 1, [10] * 5000, None, "tiles")])
def test_routes_of_reductions(artifact_cache, op, dtype, d, lengths, max_len, route):
    from gpu_helpers import check, run_program
    program = Compiler().compile(ProgramSpec(op, dtype, d, "i64"), artifact_cache)
    offsets = offsets_from_lengths(np.array(lengths, dtype=np.int64), "i64")
    values = np.random.default_rng(d).normal(size=(int(offsets[-1]), d)).astype(np.float32)
    chosen, why = program.choose(len(values), len(lengths), max_len)
    actual, report = run_program(program, values, offsets, dtype=dtype, op=op, max_len=max_len)
    assert report.selected == chosen == ("naive" if route == "naive" else "classified")
    assert bool(report.selection.get("tiles")) == bool(why.get("tiles")) == (route == "tiles")
    assert bool(report.selection.get("short_segments")) == (route == "alone")
    assert report.kernel_names[0].endswith("split_partial") == (route == "tiles")
    assert (report.classes == ("tiles",)) == (route == "tiles") and (route != "tiles" or report.thresholds == ())
    check(actual, values, offsets, op=op, dtype=dtype)
