"""GPU: one `@kernel` function called in turn with dense torch tensors, strided ones, numpy arrays and torch tensors again,
with a workspace in between (what a call keeps from the one before it: shapes, types, the workspace callback). Runs in a
process of its own that imports torch first (see tests/test_torch_adapter.py for why)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

_SCRIPT = r'''
import gc
import weakref
import numpy as np
import torch
import dvm_amd as dvm


def make():
    @dvm.kernel(ktype="mix", dynamic=True)
    def product(k, x, w):  # few tiles and a long k axis: partial tiles in the workspace
        return k.store(k.matmul(k.load(x, dvm.float16), k.load(w, dvm.float16), False, False))
    return product


f = make()
g = torch.Generator(device="cuda").manual_seed(3)
def ints(*shape):
    return torch.randint(-1, 2, shape, device="cuda", generator=g).half()
def check(got, x, w):
    got = torch.from_numpy(got).cuda() if isinstance(got, np.ndarray) else got
    assert torch.equal(got.double(), x.double() @ w.double())

kept = []
for m in (64, 8, 64):
    x, w = ints(m, 8192), ints(8192, 128)
    check(f(x, w), x, w)
    assert f.workspace_bytes() > 0 and f._ws_scratch and all(f._ws_scratch is not s for s in kept)
    kept.append(f._ws_scratch)
    wide = ints(m, 9000)
    check(f(wide[:, :8192], w), wide[:, :8192], w)
    check(f(x.cpu().numpy(), w.cpu().numpy()), x, w)
    check(f(x, w), x, w)
    f.set_workspace_allocator(lambda n: (_ for _ in ()).throw(AssertionError("not the caller's any more")))
    check(f(x, w), x, w)
s = torch.cuda.Stream()
s.wait_stream(torch.cuda.current_stream())
with torch.cuda.stream(s):
    y = f(x, w)
s.synchronize()
check(y, x, w)
gone = weakref.ref(f)
del f
assert gone() is None  # (the workspace callback holds no reference to its kernel)
print("calls in turn: ok")
'''


def test_one_kernel_called_in_turn():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root + os.pathsep + os.environ.get("PYTHONPATH", ""))
    r = subprocess.run([sys.executable, "-c", _SCRIPT], cwd=root, env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and "calls in turn: ok" in r.stdout, r.stdout + r.stderr
