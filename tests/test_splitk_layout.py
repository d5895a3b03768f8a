"""The two launches of a product whose k axis is shared, without a GPU (disassembly mode)."""
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
