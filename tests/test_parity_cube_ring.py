"""GPU parity: the matmul's tile loop on sizes whose last stage of 64 k, last rows and last columns are not whole (chunks
outside the operands are loads of nothing and read as zero). Operands are whole numbers of at most two, so every sum is exact
in fp32 and small enough for fp16, and the results must be equal."""
import numpy as np
import pytest

from dvm_amd.tester import Tester

pytestmark = pytest.mark.gpu


def _run(m, n, k, ta, tb, dtype="float16", batch=()):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a = rng.integers(-2, 3, batch + (m, k)).astype(np.float16)
    b = rng.integers(-1, 2, batch + (k, n)).astype(np.float16)
    a[..., -1, :] = 1  # the last row and column count the k that were summed
    b[..., :, -1] = 1
    t = Tester("mix")
    x, y = (np.swapaxes(a, -1, -2).copy() if ta else a), (np.swapaxes(b, -1, -2).copy() if tb else b)
    out = t.store(t.cast(t.matmul(t.load(x), t.load(y), ta, tb), "float32"))
    t.run()
    assert "fast" in t.das(), t.das()
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.abs(want).max() <= 2048  # exact in fp16
    assert np.array_equal(t.output(out).astype(np.float64), want)
    return t.das()


@pytest.mark.parametrize("tile", ["64", "128", "256"])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(8, 8, 8), (64, 64, 64), (72, 8, 56), (136, 264, 72), (256, 128, 200), (264, 520, 328), (56, 248, 520)])
def test_sizes_around_tiles_and_stages(monkeypatch, tile, ta, tb, m, n, k):
    monkeypatch.setenv("DVM_CUBE_TILE", tile)
    monkeypatch.setenv("DVM_CUBE_SPLITK", "0")
    _run(m, n, k, ta, tb)


@pytest.mark.parametrize("tile", ["64", "128", "256"])
@pytest.mark.parametrize("k", [1, 3, 63, 65, 129, 257])
def test_any_k_where_k_is_strided_in_both_operands(monkeypatch, tile, k):
    monkeypatch.setenv("DVM_CUBE_TILE", tile)
    _run(136, 264, k, True, False)


@pytest.mark.parametrize("m", [1, 7, 63, 65, 127, 130, 257])
@pytest.mark.parametrize("tb", [False, True])
def test_any_number_of_rows_and_split_k(monkeypatch, m, tb):
    for split in ("0", "3"):
        monkeypatch.setenv("DVM_CUBE_SPLITK", split)
        _run(m, 72, 456, False, tb)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_128_tile_with_two_and_with_four_stage_buffers(monkeypatch, ta, tb):
    # more tiles than compute units: two workgroups share one and each has half the local memory
    monkeypatch.setenv("DVM_CUBE_TILE", "128")
    monkeypatch.setenv("DVM_CUBE_SPLITK", "0")
    assert "lds=131072" in _run(1048, 1048, 200, ta, tb)
    assert "lds=65536" in _run(2056, 2056, 200, ta, tb)


def test_batches_end_inside_a_stage(monkeypatch):
    # the row behind the last of one matrix is the first of the next: it must not be read for it
    _run(40, 72, 88, False, True, batch=(3,))
    _run(40, 72, 88, True, False, batch=(3,))


def test_a_program_of_the_64_tile_exported_with_two_stage_buffers_still_runs():
    import ctypes
    import os
    lib = ctypes.CDLL(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dvm_amd", "lib", "libdvm_hip.so"))
    lib.dvm_hip_launch_vm_static_ws.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.POINTER(ctypes.c_uint32), ctypes.POINTER(ctypes.c_uint32),
                                                ctypes.c_uint32, ctypes.c_size_t, ctypes.c_void_p]
    lib.dvm_hip_memset.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t]
    lib.dvm_hip_synchronize_stream.argtypes = [ctypes.c_void_p]
    rng = np.random.default_rng(2)
    for m, n, k, launches in ((100, 200, 320, 1), (64, 64, 8192, 2)):
        a, b = (rng.standard_normal(s).astype(np.float16) / 16 for s in ((m, k), (k, n)))
        t = Tester("mix")
        out = t.store(t.matmul(t.load(a), t.load(b), False, False))
        t.run()
        want = t.output(out).copy()
        programs = t.programs()
        assert len(programs) == launches, t.das()
        blobs = b"".join(p[0] for p in programs)
        pairs = [v for i, p in enumerate(programs) for w in p[2] for v in (i, w)]
        words = (ctypes.c_uint32 * max(1, len(pairs)))(*pairs)
        for lds, rc in ((32768, 0), (32768 - 16, 1)):  # (1: hipErrorInvalidValue, before anything is launched)
            geo = (ctypes.c_uint32 * (3 * len(programs)))(*[v for p in programs for v in (p[1][0], p[1][1], lds)])
            assert lib.dvm_hip_memset(t.device_ptr(out), 0, want.nbytes) == 0
            got_rc = lib.dvm_hip_launch_vm_static_ws(ctypes.create_string_buffer(blobs, len(blobs)), len(programs), geo, words, len(pairs) // 2, t.workspace_bytes(), None)
            assert got_rc == rc and lib.dvm_hip_synchronize_stream(None) == 0
            got = t.output(out)
            assert np.array_equal(got.view(np.uint16), want.view(np.uint16)) if rc == 0 else not got.any()
