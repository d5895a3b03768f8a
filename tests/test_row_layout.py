"""Which layout a program that reduces the innermost axis is compiled to, without a GPU (disassembly mode): a program the
row build (vm_vector_row.hip) cannot take is what it is with that build switched off (DVM_VEC_ROW=0), word for word, and is
not cut into more launches on the way there."""
import numpy as np
import pytest

from dvm_amd.tester import Tester


def _load(t, shape, dtype):
    if dtype == "bfloat16":
        op = t.load(list(shape), dtype)
        t.input(op, np.zeros(shape, np.uint16))
        return op
    return t.load(np.zeros(shape, dtype))


def _wide(t, x, dtype):
    return x if dtype == "float32" else t.cast(x, "float32")


def rms_backward(t, rows, cols, dtype):
    x, dy, w = (_wide(t, _load(t, s, d), d) for s, d in (((rows, cols), dtype), ((rows, cols), dtype), ((cols,), "float32")))
    r = t.div(1.0, t.sqrt(t.add(t.mul(t.sum(t.mul(x, x), (1,), True), 1.0 / cols), 1e-6)))
    xh, g = t.mul(x, r), t.mul(dy, w)
    s = t.mul(t.sum(t.mul(g, xh), (1,), True), 1.0 / cols)
    dx = t.mul(t.sub(g, t.mul(xh, s)), r)
    return [dx if dtype == "float32" else t.cast(dx, dtype), t.mul(dy, xh)]


def layer_norm_backward(t, rows, cols, dtype):
    x, dy, w = (_wide(t, _load(t, s, d), d) for s, d in (((rows, cols), dtype), ((rows, cols), dtype), ((cols,), "float32")))
    mean, rstd = (_load(t, (rows, 1), "float32") for _ in range(2))
    xh, g = t.mul(t.sub(x, mean), rstd), t.mul(dy, w)
    a, b = (t.mul(t.sum(v, (1,), True), 1.0 / cols) for v in (g, t.mul(g, xh)))
    return [t.mul(t.sub(t.sub(g, a), t.mul(xh, b)), rstd), t.mul(dy, xh)]


def three_exponentials(t, rows, cols, dtype):
    a, b, c = (t.exp(_wide(t, _load(t, (rows, cols), dtype), dtype)) for _ in range(3))
    s = t.sum(t.mul(t.mul(a, b), c), (1,), True)
    return [t.div(v, s) for v in (a, b, c)]


def _compile(graph, rows, cols, dtype):
    t = Tester("split", run_mode="das")
    for o in graph(t, rows, cols, dtype):
        t.store(o)
    t.codegen()
    return t


@pytest.mark.parametrize("graph,rows,cols,dtype", [
    (rms_backward, 1, 5120, "float32"), (rms_backward, 100, 6144, "float32"), (rms_backward, 200, 8192, "float32"), (rms_backward, 200, 8192, "bfloat16"),
    (layer_norm_backward, 1, 5120, "float32"), (layer_norm_backward, 200, 8192, "float32"), (layer_norm_backward, 200, 8192, "bfloat16"),
    (three_exponentials, 1, 4096, "float32"), (three_exponentials, 256, 4096, "float32"), (three_exponentials, 4096, 4096, "bfloat16")])
def test_values_held_across_a_reduce_stay_one_launch(monkeypatch, graph, rows, cols, dtype):
    """The row build's lanes (up to twice those of the other builds) leave too few V register slots, or its slabs have none:
    the whole sub-kernel keeps the other builds' layout."""
    monkeypatch.delenv("DVM_VEC_ROW", raising=False)
    t = _compile(graph, rows, cols, dtype)
    assert t.num_launches() == 1 and " row=" not in t.das(), t.das()
    monkeypatch.setenv("DVM_VEC_ROW", "0")
    assert t.das() == _compile(graph, rows, cols, dtype).das()


def test_values_held_across_a_reduce_use_the_row_build_where_its_registers_do(monkeypatch):
    monkeypatch.delenv("DVM_VEC_ROW", raising=False)
    for graph, rows, cols in ((rms_backward, 64, 4096), (layer_norm_backward, 3, 512), (three_exponentials, 4096, 1000)):
        t = _compile(graph, rows, cols, "float32")
        assert t.num_launches() == 1 and " row=" in t.das(), t.das()
