"""GPU parity of pointwise fp32 programs whose waves hold their elements in runs of four a lane (VS_RUNS32): sizes around a wave's
512 elements, a workgroup's rounds and ragged ends, with an operand that is one element for all; a window of a tensor that
starts off 16 bytes keeps the other order. Against NumPy, to the bit."""
import numpy as np
import pytest

from dvm_amd.tester import Tester

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65527, 65529, 65536, 65537, 65543, 65544, 65545, 66040, 66047, 66048, 66049, 66559, 67080, 99999, 1 << 20, (1 << 20) + 520, 3000001])
def test_sums_and_products(n):
    rng = np.random.default_rng(n)
    x, y, one = rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32), np.array([1.25], np.float32)
    t = Tester("split")
    a, b = t.load(x), t.load(y)
    s = t.add(a, t.mul(b, t.load(one)))
    out, big, prod = t.store(s), t.store(t.maximum(s, b)), t.store(t.mul(s, a))
    t.run()
    assert (" runs " in t.das()) == (n > 65528), t.das()
    want = x + y * one
    assert np.array_equal(t.output(out), want) and np.array_equal(t.output(big), np.maximum(want, y)) and np.array_equal(t.output(prod), want * x)


@pytest.mark.parametrize("start,n", [(1, 70000), (4, 70000), (3, 66001)])
def test_a_window_of_a_tensor(start, n):
    x = np.random.default_rng(n).standard_normal(n + 8).astype(np.float32)
    t = Tester("split")
    out = t.store(t.mul(t.slice_load(x, [start], [n]), 3.0))
    t.run()
    assert np.array_equal(t.output(out), x[start:start + n] * np.float32(3.0)), t.das()


def test_a_tensor_of_another_type_keeps_the_elements_together():
    x, h = np.random.default_rng(1).standard_normal(70000).astype(np.float32), np.random.default_rng(2).standard_normal(70000).astype(np.float16)
    t = Tester("split")
    out = t.store(t.add(t.load(x), t.cast(t.load(h), "float32")))
    t.run()
    assert " runs " not in t.das(), t.das()
    assert np.array_equal(t.output(out), x + h.astype(np.float32))
