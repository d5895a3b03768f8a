"""GPU parity of the row build of the vector VM (dvm_vm_vec_row*): an output's whole reduced row lies in the registers of
its team, one to eight slabs a lane. Row lengths sit at the edges of that layout (one element more or less than a whole
number of slabs or lanes, the smallest and the longest rows, odd lengths whose rows start at every alignment), the row
counts pick few and many slabs a lane. References are float64; tolerances are the 8-element fp32 sums' (2^-24 * 3 per
sum, divided out) and the storage type's rounding."""
import numpy as np
import pytest

from dvm_amd.tester import Tester

pytestmark = pytest.mark.gpu

EPS = {"float32": 4e-6, "float16": 2e-3, "bfloat16": 1.6e-2}


def _inputs(rows, cols, dtype, seed, scale=1.0):
    x = np.random.default_rng(seed).standard_normal([rows, cols], dtype=np.float32) * np.float32(scale)
    return Tester.convert_to_bf16(x) if dtype == "bfloat16" else x.astype(dtype)


def _f64(a, dtype):
    return (Tester.convert_from_bf16(a) if dtype == "bfloat16" else a).astype(np.float64)


def _load(t, a, dtype):
    op = t.load(a.shape, dtype)
    t.input(op, a)
    return op


@pytest.mark.parametrize("rows,cols", [(3, 264), (2, 257), (5, 511), (5, 513), (70, 1000), (300, 4095), (300, 4097), (2100, 4096), (2100, 4089), (2100, 4081),
                                       (2100, 3073), (2100, 2569), (300, 12289), (9, 20001), (300, 32001), (4, 32768), (4, 32761)])
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
def test_softmax_rows(rows, cols, dtype):
    x = _inputs(rows, cols, dtype, rows * 31 + cols, 2.0)
    t = Tester("split")
    v = _load(t, x, dtype)
    v = t.cast(v, "float32") if dtype != "float32" else v
    e = t.exp(t.sub(v, t.max(v, (1,), True)))
    p = t.div(e, t.sum(e, (1,), True))
    out = t.store(t.cast(p, dtype) if dtype != "float32" else p)
    t.run()
    assert " row=" in t.das(), t.das()
    got, x64 = _f64(t.output(out), dtype), _f64(x, dtype)
    want = np.exp(x64 - x64.max(1, keepdims=True))
    want /= want.sum(1, keepdims=True)
    # (values below 1 / 16384 of a softmax are subnormal or coarse in fp16)
    assert np.allclose(got, want, rtol=EPS[dtype], atol=6e-8 if dtype == "float16" else 0)


@pytest.mark.parametrize("rows,cols", [(1, 4096), (37, 1003), (2100, 4096), (2100, 5120), (2100, 4091), (3, 16384), (6, 30000)])
def test_residual_norm_rows_with_statistics_stored(rows, cols):
    """Two 16-bit operands in one trip, a weight row, per-row outputs beside the row output."""
    x, r = _inputs(rows, cols, "float16", 1), _inputs(rows, cols, "float16", 2)
    w = np.random.default_rng(3).uniform(0.5, 1.5, [cols]).astype(np.float32)
    t = Tester("split")
    h = t.cast(t.add(_load(t, x, "float16"), _load(t, r, "float16")), "float32")
    mean = t.mul(t.sum(h, (1,), True), 1.0 / cols)
    c = t.sub(h, mean)
    var = t.mul(t.sum(t.mul(c, c), (1,), True), 1.0 / cols)
    outs = [t.store(t.mul(t.div(c, t.sqrt(t.add(var, 1e-5))), t.load(w))), t.store(mean), t.store(t.min(h, (1,), True))]
    t.run()
    assert " row=" in t.das(), t.das()
    h64 = (x + r).astype(np.float64)
    m64 = h64.mean(1, keepdims=True)
    want = (h64 - m64) / np.sqrt(h64.var(1, keepdims=True) + 1e-5) * w
    assert np.allclose(t.output(outs[0]), want, rtol=2e-5, atol=2e-6)
    assert np.allclose(t.output(outs[1]), m64, rtol=1e-5, atol=1e-7)
    assert np.array_equal(t.output(outs[2]), h64.min(1, keepdims=True).astype(np.float32))


def test_nothing_is_written_past_a_ragged_row():
    """Odd rows stored through strides into a wider buffer: what lies between them stays as it was."""
    rows, cols, pitch = 65, 1021, 1024
    x = _inputs(rows, cols, "float32", 5)
    want = np.zeros([rows, pitch], np.float32)
    want[:, :cols] = x - x.max(1, keepdims=True)
    t = Tester("split")
    v = t.load(x)
    t.view_store_expect(t.sub(v, t.max(v, (1,), True)), (pitch, 1), want, 0)
    assert t.run_check()


@pytest.mark.parametrize("b,h,cols", [(3, 5, 264), (7, 3, 1003), (2, 9, 4096), (70, 31, 513), (61, 37, 4090), (1, 6, 12289), (257, 3, 300)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_two_kept_axes(b, h, cols, dtype):
    """Rows numbered by two axes that do not merge: operands broadcast along either of them, one value per row of either, and
    the result of every row stored."""
    x, m = _inputs(b * h, cols, dtype, b * 7 + cols).reshape(b, h, cols), _inputs(b, cols, dtype, 3).reshape(b, 1, cols)
    g = _inputs(h, cols, "float32", 4).reshape(1, h, cols)
    rng = np.random.default_rng(h)
    s, o = rng.uniform(0.5, 1.5, [1, h, 1]).astype(np.float32), rng.uniform(-1.0, 1.0, [b, 1, 1]).astype(np.float32)
    t = Tester("split")
    wide = (lambda v: v) if dtype == "float32" else (lambda v: t.cast(v, "float32"))
    z = t.add(t.add(t.mul(wide(_load(t, x, dtype)), t.load(s)), wide(_load(t, m, dtype))), t.load(o))
    top = t.max(z, (2,), True)
    e = t.exp(t.sub(z, top))
    p = t.mul(t.div(e, t.sum(e, (2,), True)), t.load(g))
    outs = [t.store(p), t.store(top)]
    t.run()
    kdims = ("  kdims: %d %d" % (h, b)) if b > 1 else "  kdims: %d" % h
    assert " row=" in t.das() and kdims in t.das(), t.das()
    x64, m64 = _f64(x.reshape(b * h, cols), dtype).reshape(b, h, cols), _f64(m.reshape(b, cols), dtype).reshape(b, 1, cols)
    z32 = ((x64.astype(np.float32) * s + m64.astype(np.float32)) + o)  # (rounded operator by operator, as the program does)
    e64 = np.exp(z32.astype(np.float64) - z32.max(2, keepdims=True))
    assert np.array_equal(t.output(outs[1]), z32.max(2, keepdims=True))
    # (the difference inside exp is rounded to fp32: half a unit in the last place of at most 16)
    assert np.allclose(t.output(outs[0]), e64 / e64.sum(2, keepdims=True) * g, rtol=4e-6, atol=0)


@pytest.mark.parametrize("b,h,cols", [(5, 7, 1000), (3, 40, 1021), (50, 45, 2048)])
def test_rows_read_and_written_through_strides(b, h, cols):
    """[h, b, cols] in memory read as [b, h, cols] and the result written as [h, b, cols + 3]: both kept axes with strides of
    their own, rows that start at any element, nothing written between them."""
    x = _inputs(h * b, cols, "float32", 11).reshape(h, b, cols)
    t = Tester("split")
    v = t.view_load([b, h, cols], [cols, b * cols, 1], x)
    d = t.sub(v, t.max(v, (2,), True))
    pitch = cols + 3
    want = np.zeros([h, b, pitch], np.float32)
    want[:, :, :cols] = x - x.max(2, keepdims=True)
    t.view_store_expect(d, (pitch, b * pitch, 1), want, 0)
    assert t.run_check() and " row=" in t.das() and "  kdims: %d %d" % (h, b) in t.das(), t.das()


def _held_cases():
    # two slabs a lane: the first in whole lines, the last (ragged but for 1024) side by side; the values held across the reduce
    # lie in V registers
    return [(2100, 520), (2100, 777), (2100, 1000), (2100, 1017), (2100, 1024), (1100, 1031), (1100, 2047)]


def _assert_held(t):
    das = t.das()
    assert " row=2 " in das and "vslots=0" not in das and t.num_launches() == 1, das


@pytest.mark.parametrize("rows,cols", _held_cases())
def test_fp32_rows_with_exponentials_held_across_the_reduce(rows, cols):
    xs = [_inputs(rows, cols, "float32", 100 * cols + i, 0.5) for i in range(3)]
    t = Tester("split")
    e = [t.exp(t.load(x)) for x in xs]
    s = t.sum(t.mul(t.mul(e[0], e[1]), e[2]), (1,), True)
    outs = [t.store(t.div(v, s)) for v in e]
    t.run()
    _assert_held(t)
    e64 = [np.exp(x.astype(np.float64)) for x in xs]
    s64 = (e64[0] * e64[1] * e64[2]).sum(1, keepdims=True)
    # units in the last place: an exponential 1.2, three of them and two products 4.6, eight elements' sum 1.5, the sum's and
    # the quotient's rounding 1
    for o, v in zip(outs, e64):
        assert np.allclose(t.output(o), v / s64, rtol=8.3 * 2.0 ** -23, atol=0)


@pytest.mark.parametrize("rows,cols", _held_cases())
@pytest.mark.parametrize("centred", [False, True])
def test_fp32_rows_of_a_norms_backward(rows, cols, centred):
    x, dy = (_inputs(rows, cols, "float32", 100 * cols + i) for i in range(2))
    w = np.random.default_rng(3).uniform(0.5, 1.5, [cols]).astype(np.float32)
    x64, dy64, w64 = (a.astype(np.float64) for a in (x, dy, w))
    mean = x64.mean(1, keepdims=True).astype(np.float32) if centred else np.zeros((rows, 1), np.float32)
    rstd = (1.0 / np.sqrt(((x64 - mean) ** 2).mean(1, keepdims=True) + 1e-6)).astype(np.float32)
    t = Tester("split")
    vx, vdy, vw = t.load(x), t.load(dy), t.load(w)
    if centred:
        r = t.load(rstd)
        xh = t.mul(t.sub(vx, t.load(mean)), r)
    else:
        r = t.div(1.0, t.sqrt(t.add(t.mul(t.sum(t.mul(vx, vx), (1,), True), 1.0 / cols), 1e-6)))
        xh = t.mul(vx, r)
    g = t.mul(vdy, vw)
    b = t.mul(t.sum(t.mul(g, xh), (1,), True), 1.0 / cols)
    inner = t.sub(t.sub(g, t.mul(t.sum(g, (1,), True), 1.0 / cols)), t.mul(xh, b)) if centred else t.sub(g, t.mul(xh, b))
    dx, dw = t.store(t.mul(inner, r)), t.store(t.mul(vdy, xh))
    t.run()
    _assert_held(t)
    r64 = rstd.astype(np.float64) if centred else 1.0 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-6)
    h64, g64 = (x64 - mean) * r64, dy64 * w64
    want = (g64 - (g64.mean(1, keepdims=True) if centred else 0.0) - h64 * (g64 * h64).mean(1, keepdims=True)) * r64
    # sixteen halves of a unit in the last place of the terms' sizes: five roundings of a normalised element (of |x| + |mean|, that of the
    # root among them), four of g and the differences, five of a mean (eight elements' sum, its rounding, the factor)
    h = (np.abs(x64) + np.abs(mean)) * r64
    size = (np.abs(g64) + np.abs(g64).mean(1, keepdims=True) + h * (np.abs(g64) * h).mean(1, keepdims=True)) * r64
    assert (np.abs(t.output(dx) - want) <= 16 * 2.0 ** -24 * size).all()
    assert (np.abs(t.output(dw) - dy64 * h64) <= 8 * 2.0 ** -24 * np.abs(dy64) * h).all()
