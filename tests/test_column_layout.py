"""Which reduces over leading axes stay in one launch, without a GPU (disassembly mode): those the column build
(vm_vector_col.hip) takes. Any other is shared between workgroups, as it is with that build switched off (DVM_VEC_COL=0)."""
import re

import numpy as np
import pytest

from dvm_amd.tester import Tester


def _sum(t, x):
    return t.sum(x, (0,), False)


def plain(t, x):
    return [_sum(t, x)]


def sum_and_squares(t, x):
    return [_sum(t, x), _sum(t, t.mul(x, x))]


def beside_a_product_with_a_number(t, x):
    return [_sum(t, x), t.mul(x, 2.0)]


def beside_its_exponential(t, x):
    return [_sum(t, x), t.exp(x)]


def beside_its_cast(t, x):
    return [_sum(t, x), t.cast(x, "bfloat16")]


def beside_a_sum_with_its_rows(t, x):
    return [_sum(t, x), t.add(t.sum(x, (1,), True), x)]


def three_reduces(t, x):
    return [_sum(t, x), t.max(x, (0,), False), t.min(x, (0,), False)]


def fourth_powers(t, x):
    q = t.mul(x, x)
    return [_sum(t, t.mul(q, q))]


def _launches(graph, shape, monkeypatch, off=False, view=None):
    if off:
        monkeypatch.setenv("DVM_VEC_COL", "0")
    else:
        monkeypatch.delenv("DVM_VEC_COL", raising=False)
    t = Tester("split", run_mode="das")
    if view is None:
        x = t.load(np.zeros(shape, np.float32))
    else:
        x = t.view_load(shape, view, "float32")
        t.input(x, np.zeros(shape, np.float32))
    for o in graph(t, x):
        t.store(o)
    t.codegen()
    entries = re.findall(r"^entry.*$", t.das(), re.M)
    return entries, [int(re.search(r"blocks=(\d+)", e).group(1)) for e in entries]


@pytest.mark.parametrize("shape", [(1024, 4096), (4096, 2048), (2048, 512), (3000, 1000)])
@pytest.mark.parametrize("graph,launches", [(plain, 1), (sum_and_squares, 1), (beside_a_sum_with_its_rows, 2)])
def test_taken_by_the_column_build(graph, launches, shape, monkeypatch):
    entries, _ = _launches(graph, shape, monkeypatch)
    assert len(entries) == launches and sum(" columns " in e for e in entries) == 1, entries


@pytest.mark.parametrize("shape", [(1024, 4096), (4096, 2048), (2048, 512), (3000, 1000)])
@pytest.mark.parametrize("graph", [beside_a_product_with_a_number, beside_its_exponential, beside_its_cast, three_reduces, fourth_powers])
def test_refused_by_the_column_build(graph, shape, monkeypatch):
    entries, blocks = _launches(graph, shape, monkeypatch)
    before, blocks_before = _launches(graph, shape, monkeypatch, off=True)
    assert len(blocks) == len(blocks_before) and all(n >= b for n, b in zip(blocks, blocks_before)), (entries, before)


@pytest.mark.parametrize("graph", [plain, sum_and_squares])
def test_columns_that_are_no_line_of_memory(graph, monkeypatch):
    shape = (4096, 2048)
    entries, blocks = _launches(graph, shape, monkeypatch, view=(1, 4096))
    before, blocks_before = _launches(graph, shape, monkeypatch, off=True, view=(1, 4096))
    assert blocks == blocks_before, (entries, before)


@pytest.mark.parametrize("shape", [(6000, 1000), (5000, 1000), (9000, 1000), (4096, 12000), (300, 33000)])
def test_no_more_workgroups_than_the_chip_takes_at_once(shape, monkeypatch):
    entries, _ = _launches(plain, shape, monkeypatch)
    assert " columns " in entries[0] and int(re.search(r"items=(\d+)", entries[0]).group(1)) <= 1280, entries


def test_a_kernel_of_many_shapes(monkeypatch):
    # the refusal of one shape says nothing about another one of the same kernel
    monkeypatch.delenv("DVM_VEC_COL", raising=False)
    t = Tester("split:dyn", run_mode="das")
    x = t.load((4096, 2048), "float32")
    q = t.mul(x, x)
    t.store(_sum(t, t.mul(q, q)))
    seen = {}
    for rows in (4096, 64, 4096, 2048, 64, 4096):
        t.input(x, np.zeros((rows, 2048), np.float32))
        t.codegen()
        blocks = tuple(int(b) for b in re.findall(r"blocks=(\d+)", t.das()))
        assert seen.setdefault(rows, blocks) == blocks
        assert rows == 64 or max(blocks) >= 128, t.das()
