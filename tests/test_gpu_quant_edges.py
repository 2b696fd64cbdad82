"""The quantizer and the AWQ search where their shortcuts end: weights on and
next to rounding boundaries of their scale, empty groups, magnitudes at the ends
of the f32 range, and error sums of a chunk less, exactly and more than a chunk
(8192 terms). Codes, scales and errors equal the oracle's bit for bit."""
import numpy as np
import pytest

import oracle
from ferrolm_amd import gpu
from ferrolm_amd.weights import INT4, INT8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [INT8, INT4], ids=["int8", "int4"])
@pytest.mark.parametrize("case", ["halves", "near halves", "zeros", "tiny", "denormal", "huge", "one value"])
@pytest.mark.parametrize("weighted", [False, True])
def test_quantizer_boundaries(ctx, kind, case, weighted):
    rng = np.random.default_rng(7)
    hi = 127 if kind == INT8 else 7
    w = rng.integers(-2 * hi, 2 * hi + 1, (64, 160)).astype(np.float32) / 2  # halves of a code at scale 1
    w[:, ::32] = hi
    if case == "near halves":
        w = np.nextafter(w, np.where(rng.random(w.shape) < 0.5, -np.inf, np.inf).astype(np.float32))
    elif case == "zeros":
        w[::3] = 0
        w[:, 32:64] = 0
    elif case in ("tiny", "denormal", "huge"):
        w = w * np.float32({"tiny": 1e-33, "denormal": 1e-41, "huge": 1e36}[case])
    elif case == "one value":
        w = np.full_like(w, -0.7)
    imp = rng.random(160).astype(np.float32) if weighted else None
    got, want = gpu.quantize(ctx, kind, w, imp), oracle.quantize(kind, w, imp)
    assert np.array_equal(got.s, want.s)
    assert np.array_equal(got.q, want.q)


@pytest.mark.parametrize("rows,m", [(32, 1), (32, 255), (32, 256), (32, 257), (288, 91)])
def test_search_errors_across_chunks(ctx, rows, m):
    rng = np.random.default_rng(rows + m)
    w = (0.02 * rng.standard_normal((rows, 160))).astype(np.float32)
    cal = rng.standard_normal((m, 160)).astype(np.float32) * np.exp(2 * rng.standard_normal((m, 1))).astype(np.float32)
    got, want = gpu.awq_search(ctx, INT4, w, cal), oracle.awq_search(INT4, w, cal)
    assert got[1:4] == tuple(want[1:4])
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[4].q, want[4].q)
    assert np.array_equal(got[4].s, want[4].s)


@pytest.mark.parametrize("kind", [INT8, INT4], ids=["int8", "int4"])
@pytest.mark.parametrize("rows,cols", [(2016, 2048), (2048, 2048), (2080, 2080), (160, 32768), (160, 32800)])
def test_large_matrices_in_panels(ctx, kind, rows, cols):
    """Copied whole (under 16 MB, or panels over 4 MB) or through staging slots of
    whole panels, the last one short: a panel's codes and scales are those it
    has on its own."""
    rng = np.random.default_rng(rows)
    w = (0.02 * rng.standard_normal((rows, cols))).astype(np.float32)
    imp = rng.random(cols).astype(np.float32)
    for weight in (None, imp):
        got = gpu.quantize(ctx, kind, w, weight)
        parts = [gpu.quantize(ctx, kind, w[r : r + 32], weight) for r in range(0, rows, 32)]
        assert np.array_equal(got.q.ravel(), np.concatenate([p.q.ravel() for p in parts]))
        assert np.array_equal(got.s.ravel(), np.concatenate([p.s.ravel() for p in parts]))


def test_search_copies_a_large_matrix(ctx):
    """17 MB of weights in five slots, the last one short."""
    rng = np.random.default_rng(3)
    w = (0.02 * rng.standard_normal((2080, 2080))).astype(np.float32)
    cal = rng.standard_normal((4, 2080)).astype(np.float32)
    got, want = gpu.awq_search(ctx, INT8, w, cal), oracle.awq_search(INT8, w, cal)
    assert got[1:4] == tuple(want[1:4])
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[4].q, want[4].q)
    assert np.array_equal(got[4].s, want[4].s)


def test_search_over_more_rows_than_one_grid(ctx):
    """524,280 rows fill a launch's grid; the rest are a second one's."""
    rng = np.random.default_rng(5)
    w = (0.02 * rng.standard_normal((32, 32))).astype(np.float32)
    cal = rng.standard_normal((524_280 + 13, 32)).astype(np.float32)
    got, want = gpu.awq_search(ctx, INT8, w, cal), oracle.awq_search(INT8, w, cal)
    assert got[1:4] == tuple(want[1:4])
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[4].q, want[4].q)


@pytest.mark.parametrize("row", [0, 300, 600])
def test_search_errors_that_are_not_finite(ctx, row):
    """A calibration row whose outputs overflow, in the first, a middle and the last chunk of 8192 error terms:
    such a chunk has no map and its terms are added one by one. (The row's squares are still finite: the
    importances, and so the codes, are ordinary.)"""
    rng = np.random.default_rng(row)
    w = (1e20 * rng.standard_normal((32, 160))).astype(np.float32)
    cal = rng.standard_normal((601, 160)).astype(np.float32)
    cal[row, 7:11] = 1e19
    got, want = gpu.awq_search(ctx, INT8, w, cal), oracle.awq_search(INT8, w, cal)
    assert not np.isfinite(want[2])
    assert np.array_equal(np.float64(got[1:4]), np.float64(want[1:4]), equal_nan=True)
    assert np.array_equal(got[0], want[0])
    assert np.array_equal(got[4].s, want[4].s) and np.array_equal(got[4].q, want[4].q)
