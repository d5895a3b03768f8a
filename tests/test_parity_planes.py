"""GPU parity of the row build over two reduced axes (dvm_vm_vec_planes*): a channel's planes lie in the registers of its team,
and every slab may be the ragged last one of its plane. Planes of a few elements to whole slabs and odd ends, one to many planes
to a lane's slabs, every number of slabs a lane. References are float64; the tolerances are the 8-element fp32 sums' (2^-24 * 3
per sum, through the variance's division by its root) and the storage type's rounding."""
import numpy as np
import pytest

from dvm_amd.tester import Tester

pytestmark = pytest.mark.gpu

EPS = {"float32": 8e-6, "float16": 2e-3, "bfloat16": 1.6e-2}


def _load(t, x, dtype):
    if dtype != "bfloat16":
        return t.load(x.astype(dtype)), x.astype(dtype).astype(np.float64)
    bits = Tester.convert_to_bf16(x)
    v = t.load(bits.shape, "bfloat16")
    t.input(v, bits)
    return v, Tester.convert_from_bf16(bits).astype(np.float64)


@pytest.mark.parametrize("n,c,h,w", [(5, 7, 7, 7), (11, 300, 11, 11), (40, 3, 3, 3), (34, 5, 4, 2), (2, 43, 54, 54), (9, 427, 35, 35), (17, 30, 35, 35),
                                     (5, 52, 32, 32), (10, 6, 14, 14), (3, 2100, 31, 33), (32, 2, 1, 1023), (7, 2100, 27, 27), (2, 600, 73, 73), (31, 9, 1, 9)])
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
def test_batch_norm_over_planes(n, c, h, w, dtype):
    rng = np.random.default_rng(n * 1000 + h)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32) * 2 + 0.5
    g, b = rng.uniform(0.5, 1.5, (1, c, 1, 1)).astype(np.float32), rng.standard_normal((1, c, 1, 1)).astype(np.float32)
    t = Tester("split")
    v, x64 = _load(t, x, dtype)
    v = t.cast(v, "float32") if dtype != "float32" else v
    inv = 1.0 / (n * h * w)
    mean = t.mul(t.sum(v, (0, 2, 3), True), inv)
    d = t.sub(v, mean)
    var = t.mul(t.sum(t.mul(d, d), (0, 2, 3), True), inv)
    y = t.add(t.mul(t.div(d, t.sqrt(t.add(var, 1e-5))), t.load(g)), t.load(b))
    out, mo = t.store(t.cast(y, dtype) if dtype != "float32" else y), t.store(mean)
    t.run()
    assert n * ((h * w + 7) // 8) <= 32 or (" row=" in t.das() and t.num_launches() == 1), t.das()
    m64 = x64.mean((0, 2, 3), keepdims=True)
    want = (x64 - m64) / np.sqrt(x64.var((0, 2, 3), keepdims=True) + 1e-5) * g + b
    got = t.output(out)
    got = (Tester.convert_from_bf16(got) if dtype == "bfloat16" else got).astype(np.float64)
    assert np.allclose(got, want, rtol=EPS[dtype], atol=EPS[dtype])
    assert np.allclose(t.output(mo).astype(np.float64), m64, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("n,c,hw", [(9, 5, 49), (33, 70, 121), (6, 300, 1225), (4, 3, 8), (40, 17, 9)])
def test_extremes_over_planes_and_two_operands(n, c, hw):
    rng = np.random.default_rng(hw)
    x, r = (rng.standard_normal((n, c, hw)).astype(np.float16) for _ in range(2))
    x[0, 0, :] = -np.inf
    t = Tester("split")
    s = t.add(t.load(x), t.load(r))
    hi, lo = t.max(s, (0, 2), True), t.min(s, (0, 2), True)
    out, mx = t.store(t.sub(s, t.max(s, (0, 2), True))), t.store(t.sub(hi, lo))
    t.run()
    want = x + r
    top, low = want.max((0, 2), keepdims=True), want.min((0, 2), keepdims=True)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(t.output(out), want - top, equal_nan=True) and np.array_equal(t.output(mx), top - low, equal_nan=True), t.das()


def test_an_operand_without_one_of_the_axes_keeps_the_other_builds():
    rng = np.random.default_rng(5)
    x, pos, per = (rng.standard_normal(s).astype(np.float32) for s in ((9, 12, 35), (1, 1, 35), (9, 1, 35)))
    for other in (pos, per):
        t = Tester("split")
        v = t.mul(t.load(x), t.load(other))
        out = t.store(t.sub(v, t.mul(t.sum(v, (0, 2), True), 1.0 / (9 * 35))))
        t.run()
        assert " row=" not in t.das(), t.das()
        w = x.astype(np.float64) * other
        assert np.allclose(t.output(out), w - w.mean((0, 2), keepdims=True), rtol=4e-6, atol=4e-6)


@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 9), (5, 63), (33, 100), (4095, 64), (4095, 256), (8192, 249), (8193, 9), (4096, 64)])
def test_short_rows_with_a_wave_for_each(rows, cols):
    # (a wave for each up to 4095 rows, to 8192 where rows do not start on 16 bytes)
    x = np.random.default_rng(rows + cols).standard_normal((rows, cols)).astype(np.float32)
    t = Tester("split")
    v = t.load(x)
    e = t.exp(t.sub(v, t.max(v, (1,), True)))
    out = t.store(t.div(e, t.sum(e, (1,), True)))
    t.run()
    assert rows == 1 or (" row=1 " in t.das()) == (rows < (8193 if cols % 4 else 4096)), t.das()
    w = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
    assert np.allclose(t.output(out), w / w.sum(1, keepdims=True), rtol=4e-6)
