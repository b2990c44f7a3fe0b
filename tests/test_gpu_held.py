"""Block-per-segment softmax that holds a segment in a workgroup's registers
(csrc/held.hpp), against the oracle at its edges: segments of one row, of
exactly the rows it holds, one more (streamed), the array's end inside a
vector, and columns with -inf, NaN and only -inf; which calls take it and which
the streaming kernel; and columns of large magnitude on every softmax path."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ragged import Compiler, ProgramSpec
from ragged import native
from ragged.workloads import offsets_from_lengths

pytestmark = pytest.mark.gpu


def geometry_of(program, dtype, d):
    """(rows a workgroup holds, lanes per row, access bytes) of a program."""
    vec = program.metadata["d_vector"]
    if program.metadata["mapping"] == "flat":
        return 8 * 256 * vec // d, 1, 16
    lanes = 1
    while lanes < -(-d // vec) and lanes < 256:
        lanes *= 2
    return 16 * (256 // lanes), lanes, vec * (2 if dtype == "bf16" else 4)


def role_of(program, n, b):
    """The kernel of the program's last block-per-segment plan for (n, b)."""
    plans = [plan for key, plan in program.naive._plans.items() if key[1:3] == (n, b)]
    return plans[-1].steps[0][0]


@pytest.mark.parametrize("dtype,d", [("f32", 1), ("f32", 2), ("f32", 16), ("f32", 25), ("f32", 300), ("bf16", 1),
                                     ("bf16", 4), ("bf16", 5), ("bf16", 46), ("bf16", 64), ("bf16", 84)])
def test_held_segments(artifact_cache, dtype, d):
    from gpu_helpers import check, run_program
    program = Compiler().compile(ProgramSpec("softmax", dtype, d, "i64", scale=1.25), artifact_cache)
    held, _, access = geometry_of(program, dtype, d)
    # (The longest segment given is the one the kernel is for, whatever the
    # lengths: it streams a segment that it cannot hold.)
    most = native.held_rows(program.naive._native_spec())
    rng = np.random.default_rng(d)
    for lengths in ([1, 0, 2, held, 7], [held + 1, 3, held - 1, 0], [held] * 2 + [held // 8 + 1] * 40, [6 * held, 2]):
        offsets = offsets_from_lengths(np.array(lengths, dtype=np.int64), "i64")
        values = rng.normal(size=(int(offsets[-1]), d)).astype(np.float32) * 4
        values[rng.random(values.shape) < 0.01] = -np.inf
        values[int(offsets[-2]):, 0] = -np.inf
        values[0, d - 1] = np.nan
        for max_len in (most, max(lengths)):
            actual, report = run_program(program, values, offsets, dtype=dtype, op="softmax", select="naive",
                                         max_len=max_len)
            assert report.selected == "naive" and len(report.kernel_names) == 1
            check(actual, values, offsets, op="softmax", dtype=dtype, scale=1.25)
            if program.metadata["mapping"] == "flat":
                fits = sum(lengths) <= held * len(lengths)        # the mean
            else:
                fits = access > 2 and max_len <= most
            expected = "block" if fits else "naive"
            if sum(lengths) * 4 >= held * len(lengths):      # (not too short to pay)
                assert role_of(program, int(offsets[-1]), len(lengths)) == expected, (lengths[:4], max_len)


@pytest.mark.parametrize("dtype,d,mean,most,role", [
    ("bf16", 64, 2, 512, "block"), ("bf16", 64, 300, 513, "naive"), ("bf16", 64, 30, None, "naive"),
    ("bf16", 84, 8, 128, "block"), ("bf16", 84, 7, 128, "naive"), ("f32", 128, 8, 128, "block"),
    ("f32", 128, 7, 128, "naive"), ("f32", 500, 8, 32, "block"), ("f32", 500, 7, 32, "naive"),
    ("bf16", 46, 20, 32, "block"), ("bf16", 46, 20, 33, "naive"), ("bf16", 25, 20, 20, "naive"),
    ("bf16", 1024, 16, 16, "naive"), ("f32", 1, 3000, 8188, "block"), ("f32", 1, 3000, 9000, "block"),
    ("f32", 1, 3000, None, "block"), ("f32", 1, 8193, 8193, "naive")])
def test_segments_are_held_where_it_pays(artifact_cache, dtype, d, mean, most, role):
    """Rows: the longest segment known to fit and the mean not below a row (of
    more than 32 lanes, four rows) per thread; flat: the mean fits."""
    from gpu_helpers import run_program
    program = Compiler().compile(ProgramSpec("softmax", dtype, d, "i64"), artifact_cache)
    offsets = offsets_from_lengths(np.full(600, mean, dtype=np.int64), "i64")
    values = np.zeros((int(offsets[-1]), d), dtype=np.float32)
    actual, _ = run_program(program, values, offsets, dtype=dtype, op="softmax", select="naive", max_len=most)
    assert role_of(program, len(values), 600) == role
    assert np.allclose(actual, 1 / mean, rtol=4e-3)


def large_columns(offsets, d, rng):
    """Logits whose columns are of very large magnitude, as padding and masks
    make them: constant at -1e9, the lowest finite bf16 or 1e6, steps of an
    ulp at -1e5 and 1e6, padding among ordinary values; and an ordinary one."""
    lowest = -3.3895e38
    kinds = [lambda k: np.full(k, -1e9), lambda k: np.full(k, lowest), lambda k: np.full(k, 1e6),
             lambda k: -99840 - 512 * rng.integers(0, 2, k), lambda k: 999424 + 4096 * rng.integers(0, 2, k),
             lambda k: np.where(rng.random(k) < 0.5, lowest, rng.normal(size=k)), lambda k: 2 * rng.normal(size=k)]
    values = np.empty((int(offsets[-1]), d), dtype=np.float32)
    for s, (start, end) in enumerate(zip(offsets[:-1], offsets[1:])):
        for column in range(d):
            values[start:end, column] = kinds[(s + column) % len(kinds)](int(end - start))
    return values


@pytest.mark.parametrize("select", ["naive", "classified"])
@pytest.mark.parametrize("dtype,d", [("f32", 1), ("f32", 16), ("bf16", 1), ("bf16", 2), ("bf16", 25), ("bf16", 46),
                                     ("bf16", 64), ("bf16", 84), ("bf16", 128)])
def test_columns_of_large_magnitude(artifact_cache, dtype, d, select):
    """exp(x - max) / sum depends on x - max alone, whatever the magnitude of
    the column: short segments (held), and among them long ones (streamed;
    chunks merged by all readers and by tree)."""
    from gpu_helpers import check, run_program
    program = Compiler().compile(ProgramSpec("softmax", dtype, d, "i64"), artifact_cache)
    rng = np.random.default_rng(d)
    for lengths in ([4, 30, 1, 0, 2, 50, 7] * 7, [4, 300, 1, 0, 40, 20_000 // min(d, 16), 7] * 2):
        offsets = offsets_from_lengths(np.array(lengths, dtype=np.int64), "i64")
        values = large_columns(offsets, d, rng)
        actual, report = run_program(program, values, offsets, dtype=dtype, op="softmax", select=select,
                                     max_len=max(lengths))
        assert report.selected == select
        check(actual, values, offsets, op="softmax", dtype=dtype)


@pytest.mark.parametrize("select", ["naive", "classified"])
@pytest.mark.parametrize("dtype,d", [("f32", 16), ("bf16", 16), ("bf16", 46), ("bf16", 128)])
def test_masked_columns(artifact_cache, dtype, d, select):
    """An additive mask of -1e9 over a whole column of a segment, over part of
    one, and over none."""
    from gpu_helpers import check, run_program
    program = Compiler().compile(ProgramSpec("softmax", dtype, d, "i64", scale=0.125, mask=True), artifact_cache)
    rng = np.random.default_rng(d)
    lengths = [4, 300, 1, 0, 40, 20_000 // d, 7] * 2
    offsets = offsets_from_lengths(np.array(lengths, dtype=np.int64), "i64")
    values = 16 * rng.normal(size=(int(offsets[-1]), d)).astype(np.float32)
    mask = np.zeros_like(values)
    for s, (start, end) in enumerate(zip(offsets[:-1], offsets[1:])):
        mask[start:end, s % 3::3] = -1e9
        mask[start:end, (s + 1) % 3::3] = np.where(rng.random((end - start, len(range((s + 1) % 3, d, 3)))) < 0.5, -1e9, 0)
    actual, report = run_program(program, values, offsets, dtype=dtype, op="softmax", select=select, mask=mask,
                                 max_len=max(lengths))
    assert report.selected == select
    check(actual, values, offsets, op="softmax", dtype=dtype, mask=mask, scale=0.125)


@pytest.mark.parametrize("dtype,d", [("bf16", 46), ("bf16", 128), ("bf16", 1024)])
def test_large_columns_of_deferred_chunks(artifact_cache, dtype, d):
    """Chunks that stop waiting are re-read with the same bits."""
    from gpu_helpers import run_program
    program = Compiler().compile(ProgramSpec("softmax", dtype, d, "i64"), artifact_cache)
    offsets = offsets_from_lengths(np.array([3, 60_000 // d, 0, 400_000 // d, 5], dtype=np.int64), "i64")
    values = large_columns(offsets, d, np.random.default_rng(d))
    waited, _ = run_program(program, values, offsets, dtype=dtype, op="softmax", select="classified")
    module = program._module(0)
    module.set_spin_limit(0)
    try:
        deferred, _ = run_program(program, values, offsets, dtype=dtype, op="softmax", select="classified")
    finally:
        module.set_spin_limit(-1)
    assert np.array_equal(waited, deferred)
