"""dvm_rt_plan_stamp, without a GPU (disassembly mode): it changes with everything that may change what the next code generation
of a kernel gives or where its launches read and write, and with nothing else."""
import numpy as np
import pytest

from dvm_amd import _core
from dvm_amd.tester import Tester


@pytest.fixture
def kernel():
    t = Tester("split:dyn", run_mode="das")
    x = t.load(np.zeros((4, 16), np.float32))
    number = t.scalar()
    number.update(2.0)
    axes = t._shape_ref([1])
    y = t.mul(x, number)
    t.side = t.store(y)
    t.out = t.store(t.sum(y, axes, True))
    t.codegen()
    t.x, t.number, t.axes, t.y = x, number, axes, y
    return t


def _stamp(t):
    return _core._lib.dvm_rt_plan_stamp(t._rt)


def test_nothing_changed(kernel):
    before = _stamp(kernel)
    kernel.das(), kernel.workspace_bytes(), kernel.num_launches(), kernel.programs()
    other = Tester("split", run_mode="das")
    other.store(other.add(other.load(np.zeros((8,), np.float32)), 1.0))
    other.codegen()
    assert _stamp(kernel) == before == _stamp(kernel)


@pytest.mark.parametrize("change", [
    lambda t: t.codegen(), lambda t: t.normalize(), lambda t: t.reset(), lambda t: t.release_device_bindings(), lambda t: t.number.update(3.0),
    lambda t: t.number.update(3), lambda t: t.axes.update([0]), lambda t: t.input(t.x, np.zeros((5, 16), np.float32)),
    lambda t: t.bind_device(t.x, 0x1000, (4, 16)), lambda t: t.bind_device(t.x, 0x1000, (4, 16), strides=(32, 1)), lambda t: t.bind_device(t.side, 0x2000),
    lambda t: t.set_store_inplace(t.side), lambda t: t.set_store_temp(t.side), lambda t: t.store(t.y), lambda t: t.add(t.y, 1.0),
    lambda t: _core._lib.dvm_obj_set_view_offset(t.x._h, 4), lambda t: t.set_online_tuning(False), lambda t: t.set_lazy_tuning(False),
    lambda t: t.tuner_clear(), lambda t: [t.tuner_clear() for _ in range(256)], lambda t: [t.add(t.y, 1.0) for _ in range(256)],
    lambda t: [t.add(t.y, 1.0) for _ in range(65536)],
])
def test_every_change_shows(kernel, change):
    before = _stamp(kernel)
    change(kernel)
    assert _stamp(kernel) != before


def test_a_bound_load(kernel):
    other = Tester("split:dyn", run_mode="das")
    a = other.load(np.zeros((16,), np.float32))
    s = other.store(other.add(a, 1.0))
    b = other.load([16], "float32")
    before = _stamp(other)
    other.set_load_bind(b, s)
    assert _stamp(other) != before


def test_references_of_a_clone(kernel):
    t = Tester("split:dyn", run_mode="das")
    number, axes = t.clone(kernel, [kernel.number, kernel.axes])
    for ref, value in ((number, 7.0), (axes, [0])):
        before = _stamp(t)
        ref.update(value)
        assert _stamp(t) != before
