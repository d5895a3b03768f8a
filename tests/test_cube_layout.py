"""What products are compiled to, without a GPU (disassembly mode): the two launches of a shared k axis, and the route of the tiles."""
import re

import numpy as np
import pytest

from dvm_amd.tester import Tester


@pytest.mark.parametrize("m,n,k", [(8, 8192, 8192), (142, 1576, 3608), (300, 1000, 3000), (64, 64, 9728)])
def test_three_sums_of_parts_share_a_compute_unit(m, n, k):
    # (their kernel is built for three workgroups by its registers: local memory, 160 KB a unit with the program's 4 KB in
    # every workgroup, must not leave fewer)
    t = Tester("mix", run_mode="das")
    t.store(t.matmul(t.load(np.zeros((m, k), np.float16)), t.load(np.zeros((k, n), np.float16)), False, False))
    t.codegen()
    lds = [int(v) for v in re.findall(r"^entry.* lds=(\d+)", t.das(), re.M)]
    assert len(lds) == 2 and 3 * (lds[1] + 4096) <= 160 * 1024, t.das()


@pytest.mark.parametrize("m,n,k,ta,tb,route", [
    (256, 256, 192, False, True, "fast"), (256, 256, 200, False, True, "fast k-end"), (100, 72, 320, False, False, "fast"),
    (104, 72, 327, True, False, "fast k-end"), (100, 77, 320, False, True, "fast"), (100, 80, 320, True, True, "fast edge"),
    (100, 80, 328, True, True, "fast k-end edge"), (104, 77, 320, True, False, "guarded"), (104, 80, 327, False, True, "guarded"),
    (104, 80, 327, True, True, "guarded")])
def test_the_route_of_the_tiles(m, n, k, ta, tb, route):
    # a contiguous axis that is no multiple of eight: the leading dimension is none either, unless the operand is a window
    t = Tester("mix", run_mode="das")
    if "edge" in route:
        x = t.slice_load([k, m + 4], [0, 0], [k, m], "float16")
        t.input(x, np.zeros((k, m + 4), np.float16))
    else:
        x = t.load(np.zeros((k, m) if ta else (m, k), np.float16))
    t.store(t.matmul(x, t.load(np.zeros((n, k) if tb else (k, n), np.float16)), ta, tb))
    t.codegen()
    labels = re.search(r"^entry cube.* lds=\d+ (.*)$", t.das(), re.M).group(1).split()
    known = {"fast": "fast", "guarded": "guarded", "k-end-guarded-by-range": "k-end", "edge-by-element": "edge"}
    assert [known[v] for v in labels if v in known] == route.split(), t.das()
