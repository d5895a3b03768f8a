"""Which layout a program that reduces the innermost axis is compiled to, without a GPU (disassembly mode): a program the
row build (vm_vector_row.hip) cannot take is what it is with that build switched off (DVM_VEC_ROW=0), word for word, and is
not cut into more launches on the way there."""
import ctypes
import os
import re
import struct

import numpy as np
import pytest

import dvm_amd
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


def _dynamic(graph, shapes, dtype):
    """The disassembly of each of `shapes` out of one dynamic kernel, code generated twice for each."""
    t = Tester("split:dyn", run_mode="das")
    x = t.load([-1, -1], dtype)
    outs = [t.store(o) for o in graph(t, x)]
    das = []
    for shape in shapes:
        t.input(x, np.zeros(shape, np.uint16 if dtype == "bfloat16" else dtype))
        t.codegen()
        t.codegen()
        das.append(re.sub(r"@0x\w+", "@", t.das()))  # (the made-up addresses depend on what was bound before)
    assert outs
    return das


def _held_over(t, x):  # eight slabs a lane have no V registers for the three values held across the reduce
    h = t.cast(x, "float32")
    a, b, c = t.exp(h), t.exp(t.mul(h, 0.5)), t.exp(t.mul(h, 0.25))
    s = t.sum(t.mul(t.mul(a, b), c), (1,), True)
    return [t.div(v, s) for v in (a, b, c)]


def test_a_layout_that_does_not_fit_is_tried_once(monkeypatch, capfd):
    monkeypatch.setenv("DVM_DEBUG", "1")
    monkeypatch.delenv("DVM_VEC_ROW", raising=False)
    shapes = [(4096, 4096), (3, 1000), (8192, 4096), (4000, 4104), (4096, 4096)]
    many = _dynamic(_held_over, shapes, "bfloat16")
    assert capfd.readouterr().err.count("leaves the row build") == 1
    assert " row=" not in many[0] and " row=" in many[1] and " row=" not in many[2]
    # ... and what a shape compiles to does not depend on the shapes before it
    for shape, das in zip(shapes, many):
        assert _dynamic(_held_over, [shape], "bfloat16") == [das]


@pytest.mark.parametrize("op", ["sqrt", "log", "floor"])
def test_reduces_over_operators_the_row_build_has_not_are_not_tried(monkeypatch, capfd, op):
    monkeypatch.setenv("DVM_DEBUG", "1")
    das = _dynamic(lambda t, x: [t.sum(getattr(t, op)(x), (1,), True)], [(4096, 4096), (200, 1000)], "float32")
    assert "leaves the row build" not in capfd.readouterr().err
    assert all("reduce-x" in d and " row=" not in d for d in das)
    # (of one value per row they are the build's)
    das = _dynamic(lambda t, x: [getattr(t, op)(t.sum(t.abs(x), (1,), True))], [(4096, 4096)], "float32")
    assert " row=" in das[0]


# ---- imported programs: the launch check takes the row build's vocabulary and nothing else ----

END, LDS, LDI, STR, STS, ST, UN, CAST, RED, SWEEP, ENDSWEEP, FIN, LD, BINF, CMP = 0, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 16, 17, 19  # isa_gfx950.h
IMM, MEM, SREG, SREG2, REG = 1, 2, 4, 5, 0
PRE_SREG = 1 << 31


def _word(op, sub=0, kind=0, rnd=0, a=0, imm=0, ends=False):
    return op | (0x80 if ends else 0) | sub << 8 | kind << 16 | rnd << 20 | a << 24 | imm << 32


def _launch_status(blob, geometry):
    """What dvm_hip_launch_vm says of a blob on a machine without a GPU: 1 (hipErrorInvalidValue) if it refuses it, another
    error where it would have launched it."""
    lib = ctypes.CDLL(os.path.join(os.path.dirname(dvm_amd.__file__), "lib", "libdvm_hip.so"))
    return lib.dvm_hip_launch_vm(blob, *(ctypes.c_uint32(g) for g in geometry), None)


def _row_program(graph, rows, cols):
    (blob, geometry, _), = _compile(graph, rows, cols, "float32").programs()
    row_code, = struct.unpack_from("<I", blob, 72)  # VVecHeader::row_code
    off, n = row_code & 0xffff, row_code >> 16
    assert n > 0 and geometry[2] <= 64 * 1024  # (the check knows the device's local memory only with a device)
    return blob, geometry, list(struct.unpack_from("<%dQ" % n, blob, 8 * off)), off


def _with_words(blob, off, words):
    b = bytearray(blob)
    struct.pack_into("<%dQ" % len(words), b, 8 * off, *words)
    struct.pack_into("<I", b, 72, off | len(words) << 16)
    return bytes(b)


@pytest.mark.skipif(dvm_amd.Device.available(), reason="the made-up addresses of these programs must not reach a GPU")
@pytest.mark.parametrize("graph,rows,cols", [(three_exponentials, 3, 512), (rms_backward, 3, 1000), (layer_norm_backward, 2100, 512)])
def test_the_launch_check_takes_the_row_builds_vocabulary_and_nothing_else(monkeypatch, graph, rows, cols):
    monkeypatch.delenv("DVM_VEC_ROW", raising=False)
    blob, geometry, words, off = _row_program(graph, rows, cols)
    assert _launch_status(blob, geometry) != 1 and _launch_status(_with_words(blob, off, words), geometry) != 1
    n_vslot, = struct.unpack_from("<I", blob, 60)
    first_sweep = next(i for i, w in enumerate(words) if w & 0x7f == SWEEP)

    def status(in_sweep, *inserted):
        at = first_sweep + 1 if in_sweep else first_sweep
        return _launch_status(_with_words(blob, off, words[:at] + list(inserted) + words[at:]), geometry)

    taken = [(True, _word(UN, 3)), (True, _word(UN, 1)), (False, _word(UN, 8)), (True, _word(CAST, 2, rnd=2)), (True, _word(BINF, 7, IMM)), (False, _word(CMP, 5, IMM)),
             (True, _word(BINF, 0, SREG, a=7)), (False, _word(STS, a=7)), (True, _word(BINF, 3, SREG2, a=0, imm=7 | 7 << 8 | 2 << 16)),
             (True, _word(BINF, 0, REG, a=n_vslot - 2)), (False, _word(LDI))]
    for in_sweep, w in taken:
        assert status(in_sweep, w) != 1, hex(w)
    refused = [(True, _word(UN, 0)), (True, _word(UN, 2)), (True, _word(UN, 9)), (False, _word(UN, 9)),  # sqrt, log and int32 abs of a row
               (True, _word(CAST, 0)), (False, _word(CAST, 3)), (True, _word(CAST, 2, rnd=3)),             # conversions, no such rounding
               (True, _word(BINF, 8, IMM)), (False, _word(BINF, 10, IMM)), (True, _word(BINF, 0, 6)),      # logical, power, no such source
               (True, _word(BINF, 0, SREG, a=8)), (False, _word(STS, a=8)), (True, _word(LDS, a=8)),
               (True, _word(BINF, 3, SREG2, a=0, imm=8)), (True, _word(BINF, 3, SREG2, a=0, imm=8 << 8)), (True, _word(BINF, 0, REG, a=n_vslot - 1)),
               (False, _word(CMP, 8, IMM)), (False, _word(CMP, 6, IMM)), (False, _word(ENDSWEEP)), (False, _word(ENDSWEEP, ends=True)), (True, _word(ENDSWEEP)),
               (True, _word(RED, 3)), (True, _word(RED, 0x20)), (True, _word(RED, 0x11)), (True, _word(RED, 0x40, a=1)), (True, _word(RED, 0, a=2)),
               (False, _word(FIN, a=2)), (False, _word(FIN, 0x20)), (False, _word(SWEEP, imm=3 | 15 << 4)),
               (True, _word(BINF, 0, MEM, imm=PRE_SREG | 8)), (True, _word(BINF, 0, MEM, imm=PRE_SREG | 8 << 8))]
    for in_sweep, w in refused:
        assert status(in_sweep, w) == 1, hex(w)


def test_rows_that_start_inside_an_element_keep_to_the_generic_kernel(monkeypatch):
    """Packed memory with an operand at an odd byte: taken as before the row build existed, by the generic kernel at the same
    geometry; bound to an element's address again, the kernel runs on the row build again."""
    monkeypatch.delenv("DVM_VEC_ROW", raising=False)
    t = Tester("split:dyn", run_mode="das")
    x = t.load([-1, -1], "float32")
    t.store(t.div(t.exp(x), t.sum(t.exp(x), (1,), True)))
    for at, row in ((0x100000, True), (0x100004, True), (0x100002, False), (0x100001, False), (0x100004, True)):
        t.bind_device(x, at, (2100, 1000))
        t.codegen()
        (blob, geometry, _), = t.programs()
        sched, = struct.unpack_from("<I", blob, 4)
        assert ((sched & 0xf00) != 0) == row == (" row=" in t.das()) and not (at & 15 and sched & 0x20), t.das()
        if not dvm_amd.Device.available():
            assert _launch_status(blob, geometry) != 1


def _softmax(t, rows, cols, dtype):
    v = _wide(t, _load(t, (rows, cols), dtype), dtype)
    e = t.exp(t.sub(v, t.max(v, (1,), True)))
    return [t.div(e, t.sum(e, (1,), True))]


def _row_sum(t, rows, cols, dtype):
    return [t.sum(_wide(t, _load(t, (rows, cols), dtype), dtype), (1,), True)]


@pytest.mark.parametrize("graph,rows,cols,dtype,slabs,lanes", [
    (_softmax, 37, 4096, "float32", 1, 512), (_softmax, 1034, 7680, "bfloat16", 4, 256), (_softmax, 1068, 13440, "bfloat16", 4, 448),
    (_softmax, 2340, 7168, "float32", 4, 256), (_softmax, 2048, 32001, "float32", 4, 1024), (_softmax, 8192, 4096, "float32", 8, 256),
    (_softmax, 4096, 16384, "float32", 8, 256), (_softmax, 700, 17920, "float32", 3, 768), (_softmax, 5000, 2560, "float32", 5, 256),
    # a row that is read once: in rounds where a compute unit would hold one or two rows, more than two passes over the chip
    (_row_sum, 1297, 12928, "float16", 0, None), (_row_sum, 589, 28444, "float32", 0, None), (_row_sum, 500, 28444, "float32", 4, 896),
    (_row_sum, 589, 28443, "float32", 4, 896), (_row_sum, 589, 28444, "float16", 4, 896), (_row_sum, 2692, 6232, "float32", 4, 256)])
def test_slabs_and_lanes_of_a_row(monkeypatch, graph, rows, cols, dtype, slabs, lanes):
    """The layout that keeps the most rows on a compute unit (ChooseRow in schedule.cc)."""
    monkeypatch.delenv("DVM_VEC_ROW", raising=False)
    das = _compile(graph, rows, cols, dtype).das()
    assert (" row=%d " % slabs in das and " threads=%d " % lanes in das) if slabs else " row=" not in das, das


@pytest.mark.parametrize("slabs,waves,groups", [(1, 2, 10), (1, 13, 1), (2, 3, 6), (2, 4, 5), (2, 7, 2), (3, 3, 5), (3, 5, 2), (3, 9, 1), (4, 4, 4), (4, 6, 2),
                                                (4, 7, 2), (4, 8, 2), (4, 16, 1), (5, 2, 6), (5, 3, 4), (5, 4, 3), (5, 5, 1), (5, 6, 1), (6, 3, 2), (6, 5, 1), (8, 2, 4), (8, 4, 2), (8, 8, 1)])
def test_workgroups_a_compute_unit_holds(slabs, waves, groups):
    """The grid is what is resident at once: a workgroup of more than four waves needs ceil(waves / 4) of a SIMD's places."""
    lib = ctypes.CDLL(os.path.join(os.path.dirname(dvm_amd.__file__), "lib", "libdvm_hip.so"))
    lib.dvm_hip_select_block_thread.restype = ctypes.c_uint64
    lib.dvm_hip_select_block_thread.argtypes = [ctypes.c_uint64, ctypes.c_uint64, ctypes.c_uint64, ctypes.c_uint32]
    one = lib.dvm_hip_select_block_thread(1 | 8 << 8, 1 << 30, 512, 1024) >> 32  # (eight waves of eight slabs: one workgroup a unit)
    assert lib.dvm_hip_select_block_thread(1 | slabs << 8, 1 << 30, 64 * waves, 512 * waves) >> 32 == groups * one
