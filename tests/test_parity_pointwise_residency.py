"""GPU parity: pointwise programs whose V registers decide how many workgroups are resident, at sizes around a workgroup's
item (512 groups of eight elements), a full grid and a second pass; exact in float32 (every operator rounds once)."""
import numpy as np
import pytest

from dvm_amd.tester import Tester

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("held", [1, 2, 4])
@pytest.mark.parametrize("n", [1, 4095, 4096, 4097, 3 * 256 * 4096 + 8, 1024 * 4096 - 1])
def test_values_held_across_loads(held, n):
    # `held` sums that are all needed again behind the last load; operands of small whole numbers: every result is exact
    rng = np.random.default_rng(n + held)
    xs = [rng.integers(-8, 9, n).astype(np.float32) for _ in range(held + 1)]
    t = Tester("split")
    ls = [t.load(x) for x in xs]
    vals = [t.add(t.mul(ls[i], 2.0), ls[i + 1]) for i in range(held)]
    want = [xs[i] * 2 + xs[i + 1] for i in range(held)]
    total, w = vals[0], want[0]
    for v, u in zip(vals[1:], want[1:]):
        total, w = t.sub(t.mul(total, 0.5), v), w * np.float32(0.5) - u
    outs = [t.store(total)] + [t.store(v) for v in vals[1:]]
    t.run()
    for o, u in zip(outs, [w] + want[1:]):
        assert np.array_equal(t.output(o), u)
