"""GPU parity: the sum of the partial tiles of a shared k axis, which takes tiles of any size in pieces of 64 x 64. Operands
are whole numbers of at most two, so every sum and every result is exact in fp16 and fp32 and the results must be equal."""
import numpy as np
import pytest

from dvm_amd.tester import Tester

pytestmark = pytest.mark.gpu


def _ints(rng, *shape):
    return rng.integers(-1, 2, shape).astype(np.float16)


@pytest.mark.parametrize("tile,waves", [("256", "8"), ("256", "4"), ("128", "8"), ("64", "8")])
@pytest.mark.parametrize("m,n", [(1, 64), (9, 72), (33, 257), (64, 64), (65, 130), (257, 256), (300, 520), (513, 300)])
@pytest.mark.parametrize("trans", [(False, False), (True, False), (False, True)])
def test_pieces_of_ragged_tiles(monkeypatch, tile, waves, m, n, trans):
    # one row, one row past a group of eight, a fragment, a piece, a tile; bias and an activation-free store, and an
    # epilogue that goes through the interpreter
    monkeypatch.setenv("DVM_CUBE_TILE", tile)
    monkeypatch.setenv("DVM_CUBE_WAVES", waves)
    monkeypatch.setenv("DVM_CUBE_SPLITK", "5")
    k = 640
    rng = np.random.default_rng(m * 1000 + n)
    a, b, bias = _ints(rng, m, k), _ints(rng, k, n), _ints(rng, n)
    t = Tester("mix")
    p = t.matmul(t.load(a.T.copy() if trans[0] else a), t.load(b.T.copy() if trans[1] else b), *trans)
    out = t.store(t.cast(t.maximum(t.add(t.cast(p, "float32"), t.load(bias.astype(np.float32))), 0.0), "float16"))
    t.run()
    assert "split-k sum of 5" in t.das(), t.das()
    want = np.maximum(a.astype(np.float64) @ b.astype(np.float64) + bias, 0)
    assert np.array_equal(t.output(out).astype(np.float64), want)


@pytest.mark.parametrize("tile,waves", [("256", "8"), ("256", "4"), ("128", "8"), ("64", "8")])
@pytest.mark.parametrize("parts", ["2", "4", "9"])
def test_pieces_of_a_transposed_window(monkeypatch, tile, waves, parts):
    # A stored [k][m] with m no multiple of eight inside rows that are: its ragged tiles are not moved back inside the
    # output when the partials are computed, so they must not be when they are summed either
    monkeypatch.setenv("DVM_CUBE_TILE", tile)
    monkeypatch.setenv("DVM_CUBE_WAVES", waves)
    monkeypatch.setenv("DVM_CUBE_SPLITK", parts)
    k, m, n, cap = 1152, 301, 328, 304
    rng = np.random.default_rng(int(parts))
    a, b = _ints(rng, k, cap), _ints(rng, k, n)
    t = Tester("mix")
    out = t.store(t.matmul(t.slice_load(a, [0, 0], [k, m]), t.load(b), True, False))
    t.run()
    assert "split-k sum of " + parts in t.das() and "fast" in t.das(), t.das()
    assert np.array_equal(t.output(out).astype(np.float64), a[:, :m].T.astype(np.float64) @ b.astype(np.float64))


@pytest.mark.parametrize("parts", [2, 3, 4, 5, 6, 7, 8, 11])
@pytest.mark.parametrize("m", [8, 15, 17, 24, 25, 32, 40, 57])
def test_pieces_by_number_of_parts_and_groups_of_rows(monkeypatch, m, parts):
    # whole fours of parts and each remainder, one to four groups of eight rows in a fragment and none
    monkeypatch.setenv("DVM_CUBE_TILE", "64")
    monkeypatch.setenv("DVM_CUBE_SPLITK", str(parts))
    k, n = 64 * parts, 136
    rng = np.random.default_rng(m * 100 + parts)
    a, b = _ints(rng, m, k), _ints(rng, k, n)
    t = Tester("mix")
    out = t.store(t.matmul(t.load(a), t.load(b), False, False))
    t.run()
    assert "split-k sum of %d " % parts in t.das(), t.das()
    assert np.array_equal(t.output(out).astype(np.float64), a.astype(np.float64) @ b.astype(np.float64))
