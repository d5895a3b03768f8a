"""GPU parity of the column build (VS_COLS): reduces over the outer axis of a load, on the numbers of rows and columns around
what a lane, a workgroup's line of columns and a batch of rows in flight hold, against NumPy in float64 (sums: the fp64 partials
are rounded to fp32 once, half a unit in the last place) and exactly (max, min)."""
import numpy as np
import pytest

from dvm_amd.tester import Tester

pytestmark = pytest.mark.gpu


def _close(got, want):
    return (np.abs(got.astype(np.float64) - want) <= 2.0 ** -23 * np.abs(want) + 1e-30).all()


def _load(t, x, dtype):
    if dtype != "bfloat16":
        return t.load(x.astype(dtype)), x.astype(dtype).astype(np.float64)
    bits = Tester.convert_to_bf16(x)
    v = t.load(bits.shape, "bfloat16")
    t.input(v, bits)
    return v, Tester.convert_from_bf16(bits).astype(np.float64)


@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
@pytest.mark.parametrize("rows", [1, 2, 7, 64, 65, 129, 1025, 4096])
@pytest.mark.parametrize("cols", [8, 9, 15, 33, 64, 72, 129, 584, 1001])
def test_sum_of_columns(dtype, rows, cols):
    if rows == 1:
        cols += 1  # (a column of one element is no reduce)
    x = np.random.default_rng(rows * 1000 + cols).standard_normal((rows, cols)).astype(np.float32)
    t = Tester("split")
    v, x64 = _load(t, x, dtype)
    out = t.store(t.sum(t.cast(v, "float32"), (0,), False))
    t.run()
    assert rows == 1 or " columns " in t.das(), t.das()
    assert t.num_launches() == 1, t.das()
    assert _close(t.output(out), x64.sum(0))


@pytest.mark.parametrize("dtype", ["float32", "float16"])
@pytest.mark.parametrize("rows,cols", [(3, 8), (100, 37), (489, 824), (4096, 40), (2048, 2056)])
def test_two_reduces_of_a_load_and_the_arithmetic_behind_them(dtype, rows, cols):
    x = np.random.default_rng(rows + cols).standard_normal((rows, cols)).astype(dtype)
    t = Tester("split")
    v = t.load(x)
    hi, lo = t.store(t.max(v, (0,), True)), t.store(t.min(v, (0,), True))
    t.run()
    assert " columns " in t.das() and t.num_launches() == 1, t.das()
    assert np.array_equal(t.output(hi), x.max(0, keepdims=True)) and np.array_equal(t.output(lo), x.min(0, keepdims=True))
    t = Tester("split")
    v = t.cast(t.load(x), "float32")
    s, q = t.store(t.mul(t.sum(v, (0,), True), 0.5)), t.store(t.cast(t.sum(t.mul(v, v), (0,), True), "bfloat16"))
    t.run()
    assert " columns " in t.das() and t.num_launches() == 1, t.das()
    x64 = x.astype(np.float64)
    assert _close(t.output(s), 0.5 * x64.sum(0, keepdims=True))
    sq = (x.astype(np.float32) * x.astype(np.float32)).astype(np.float64).sum(0, keepdims=True)
    assert np.allclose(Tester.convert_from_bf16(t.output(q)).astype(np.float64), sq, rtol=2.0 ** -8)


@pytest.mark.parametrize("rows,cols", [(5000, 24), (9000, 136), (70001, 65)])
def test_columns_in_parts(rows, cols):
    # more rows than one launch takes: the parts are a kept axis of their own, the partial sums scattered with the parts innermost
    x = np.random.default_rng(rows).standard_normal((rows, cols)).astype(np.float32)
    t = Tester("split")
    out = t.store(t.sum(t.load(x), (0,), False))
    t.run()
    assert np.allclose(t.output(out).astype(np.float64), x.astype(np.float64).sum(0), rtol=1e-6, atol=1e-4), t.das()


def test_a_window_of_columns_that_starts_off_16_bytes():
    x = np.random.default_rng(3).standard_normal((300, 101)).astype(np.float32)
    t = Tester("split")
    out = t.store(t.sum(t.slice_load(x, [7, 5], [250, 43]), (0,), False))
    t.run()
    assert " columns " in t.das(), t.das()
    assert _close(t.output(out), x[7:257, 5:48].astype(np.float64).sum(0))


def test_nan_and_infinities_in_columns():
    x = np.random.default_rng(4).standard_normal((130, 40)).astype(np.float32)
    x[17, 3], x[60, 5], x[61, 6] = np.nan, np.inf, -np.inf
    x[:, 9] = np.finfo(np.float32).min
    t = Tester("split")
    v = t.load(x)
    hi, lo = t.store(t.max(v, (0,), False)), t.store(t.min(v, (0,), False))
    t.run()
    assert np.array_equal(t.output(hi), x.max(0), equal_nan=True) and np.array_equal(t.output(lo), x.min(0), equal_nan=True)
