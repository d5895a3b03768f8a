"""GPU: repeated calls of `@kernel` functions on torch tensors, which are made natively from the plan of the second one: new
tensors, other addresses, shapes, strides, numbers and streams from call to call, and whatever else changes the kernel in
between, against torch. Runs in a process of its own that imports torch first (see tests/test_torch_adapter.py for why)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

_SCRIPT = r'''
import numpy as np
import torch
import dvm_amd as dvm
from dvm_amd import _core

gen = torch.Generator(device="cuda").manual_seed(5)
def rnd(*shape):
    return torch.randn(shape, device="cuda", generator=gen)

@dvm.kernel(ktype="split", dynamic=True)
def axpy(k, x, y, a):
    x, y = k.load(x, dvm.float32), k.load(y, dvm.float32)
    s = k.add(k.mul(x, k.scalar(a)), y)
    return k.store(s), k.store(k.sub(s, y))

def check(x, y, a):
    s, d = axpy(x, y, a)
    want = x * a + y
    assert s.shape == want.shape and s.is_contiguous() and torch.allclose(s, want, rtol=1e-6, atol=1e-6)
    assert torch.allclose(d, want - y, rtol=1e-6, atol=1e-6)
    return s, d

def natively():  # whether a call like the last one would go through the plan
    return bool(axpy._plan)

for n in (1000, 1000, 1000, 37, 37, 1000, 1000, 1000):
    for a in (2.0, 2.0, -3.5, -3.5):
        check(rnd(n, 24), rnd(n, 24), a)
assert natively()
# what the plan recorded is told apart from everything else
p = axpy._plan
x, y = rnd(1000, 24), rnd(1000, 24)
check(x, y, -3.5); check(x, y, -3.5)
call = lambda *args: p.call(axpy, args, torch._C._cuda_getCurrentRawStream)
assert call(x, y, -3.5) is not None
for other in ((x, y, 2.0), (x, y, -3), (x[:999], y[:999], -3.5), (x.double(), y, -3.5), (x.cpu(), y, -3.5), (x, y), (x, y.t().contiguous().t(), -3.5)):
    assert call(*other) is None, other
keep = [check(x + i, y, -3.5) for i in range(4)]  # results of earlier calls stay
for i, (s, d) in enumerate(keep):
    assert torch.allclose(s, (x + i) * -3.5 + y, rtol=1e-6, atol=1e-6)
# tensors that start inside a line, on 4 and on 16 bytes
big = rnd(2, 1000 * 24 + 64)
for off in (0, 1, 4, 3, 0):
    check(big[0, off:off + 24000].view(1000, 24), big[1, off:off + 24000].view(1000, 24), -3.5)
# strided views, then dense ones of the same shape
wide = rnd(1000, 48)
for _ in range(3):
    check(wide[:, :24], y, -3.5)
for _ in range(3):
    check(x, y, -3.5)
# numpy in between, a kernel whose bindings were taken away, out=, an error
s = axpy(x.cpu().numpy(), y.cpu().numpy(), -3.5)[0]
assert np.allclose(s, (x * -3.5 + y).cpu().numpy(), rtol=1e-6, atol=1e-6)
for _ in range(3):
    check(x, y, -3.5)
axpy.release_device_bindings()
check(x, y, -3.5)
outs = [torch.empty_like(x), torch.empty_like(x)]
axpy(x, y, -3.5, out=outs)
assert torch.allclose(outs[0], x * -3.5 + y, rtol=1e-6, atol=1e-6)
try:
    axpy(x.double(), y, -3.5)
    raise SystemExit("a double went through")
except TypeError as e:
    assert "float64" in str(e)
try:
    torch.vmap(lambda v: axpy(v, y, -3.5)[0])(x.expand(2, 1000, 24))
    raise SystemExit("a batched tensor went through")
except RuntimeError:
    pass
check(x, y, -3.5)
# a workspace and two streams: every call has memory of its own
@dvm.kernel(ktype="mix", dynamic=True)
def product(k, x, w):
    return k.store(k.matmul(k.load(x, dvm.float16), k.load(w, dvm.float16), False, False))

def ints(*shape):
    return torch.randint(-1, 2, shape, device="cuda", generator=gen).half()
pairs = [(ints(64, 8192), ints(8192, 128)) for _ in range(6)]
side = torch.cuda.Stream()
side.wait_stream(torch.cuda.current_stream())
got = []
for i, (a, b) in enumerate(pairs):
    with torch.cuda.stream(side if i % 2 else torch.cuda.current_stream()):
        got.append(product(a, b))
torch.cuda.synchronize()
assert product.workspace_bytes() > 0 and bool(product._plan)
for (a, b), c in zip(pairs, got):
    assert torch.equal(c.double(), a.double() @ b.double())
# captured into a graph and replayed on new inputs
a, b = pairs[0]
static = a.clone()
g = torch.cuda.CUDAGraph()
product(static, b); product(static, b)
torch.cuda.synchronize()
with torch.cuda.graph(g):
    c = product(static, b)
for src, _ in pairs:
    static.copy_(src)
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(c.double(), src.double() @ b.double())
    assert torch.equal(product(src, b), c)
print("plans: ok")
'''

_CHANGES = r'''
import torch
import dvm_amd as dvm
from dvm_amd import _core

gen = torch.Generator(device="cuda").manual_seed(6)
def rnd(*shape):
    return torch.randn(shape, device="cuda", generator=gen)

# a store that is no result, bound by the caller, and a number that is no argument
held = {}
@dvm.kernel(ktype="split", dynamic=True)
def scaled(k, x):
    held["factor"] = _core.Kernel.scalar(k)
    held["factor"].update(2.0)
    y = k.mul(k.load(x, dvm.float32), held["factor"])
    held["side"] = k.store(k.add(y, 1.0))
    return k.store(y)

sides = [torch.zeros(40, 16, device="cuda") for _ in range(3)]
expect = [torch.zeros(40, 16) for _ in range(3)]
for turn, (side, factor) in enumerate([(0, 2.0), (0, 2.0), (0, 2.0), (0, 2.0), (1, 2.0), (1, 2.0), (1, 2.0), (1, 5.0), (1, 5.0), (1, 5.0), (2, 3.0), (0, 3.0)]):
    scaled.bind_device(held["side"], sides[side].data_ptr())
    held["factor"].update(factor)
    x = rnd(40, 16)
    got = scaled(x)
    expect[side] = (x * factor + 1.0).cpu()
    assert torch.equal(got, x * factor), turn
    for s, e in zip(sides, expect):
        assert torch.allclose(s.cpu(), e, rtol=1e-6, atol=1e-6), turn
# the same without touching anything in between: the plan makes the calls
for turn in range(4):
    x = rnd(40, 16)
    assert torch.equal(scaled(x), x * 3.0)
    assert torch.allclose(sides[0], x * 3.0 + 1.0, rtol=1e-6, atol=1e-6)
assert bool(scaled._plan)
print("changes: ok")
'''

_NUMBERS = r'''
import numpy as np
import torch
import dvm_amd as dvm

@dvm.kernel(ktype="split", dynamic=True)
def step(k, p, g, lr):
    return k.store(k.sub(k.load(p, dvm.float32), k.mul(k.load(g, dvm.float32), k.scalar(lr))))

class Counting:  # the plan, and how often it is recorded and makes a call
    def __init__(self, plan):
        self.plan, self.recorded, self.called = plan, 0, 0
        self.hold, self.release = plan.hold, plan.release
    def repeats(self, args):
        return self.plan.repeats(args)
    def record(self, *args):
        self.recorded += 1
        return self.plan.record(*args)
    def call(self, *args):
        r = self.plan.call(*args)
        self.called += r is not None
        return r

p, g = torch.randn(100, 8, device="cuda"), torch.randn(100, 8, device="cuda")
def go(lr):
    assert torch.allclose(step(p, g, lr), p - g * float(lr), rtol=1e-6, atol=1e-6)
go(0.5)
step._plan = Counting(step._plan)
# another number at every call, a number of another type, NaN among them: nothing is recorded
for i in range(20):
    go(1.0 / (1 + i))
for lr in (np.float32(0.25), np.float32(0.25), np.float64(0.25), True, True, 1, True, 0.25):
    go(lr)
assert step._plan.recorded == 0 and step._plan.called == 0
# a number that stays: recorded at its second call, made from the plan from the third on
for i in range(5):
    go(0.125)
assert step._plan.recorded == 1 and step._plan.called == 3
# and when it changes once more
go(0.25); go(0.25); go(0.25)
assert step._plan.recorded == 2 and step._plan.called == 4
# two shapes in turn: nothing is recorded, nothing is mixed up
q, h = torch.randn(7, 8, device="cuda"), torch.randn(7, 8, device="cuda")
for i in range(6):
    a, b = ((p, g), (q, h))[i % 2]
    assert torch.allclose(step(a, b, 0.25), a - b * 0.25, rtol=1e-6, atol=1e-6)
assert step._plan.recorded <= 3
print("numbers: ok")
'''


def test_numbers_that_change_are_not_recorded():
    _run(_NUMBERS, "numbers: ok")

_THREADS = r'''
import ctypes
import threading
import time
import torch
import dvm_amd as dvm

@dvm.kernel(ktype="split", dynamic=True)
def scale(k, x, a):
    return k.store(k.mul(k.load(x, dvm.float32), k.scalar(a)))

@dvm.kernel(ktype="mix", dynamic=True)
def product(k, x, w):  # (a workspace per call)
    return k.store(k.matmul(k.load(x, dvm.float16), k.load(w, dvm.float16), False, False))

x = torch.arange(4096.0, device="cuda").view(64, 64)
a = torch.randint(-1, 2, (64, 8192), device="cuda").half()
b = torch.randint(-1, 2, (8192, 128), device="cuda").half()
want = a.double() @ b.double()
for _ in range(4):
    scale(x, 2.0); product(a, b)
torch.cuda.synchronize()
assert bool(scale._plan) and product.workspace_bytes() > 0

# other threads run while a plan allocates and launches: a plan whose launch is a sleep of the C library
beats, stop = [0], threading.Event()
def beat():
    while not stop.is_set():
        beats[0] += 1
t = threading.Thread(target=beat)
t.start()
libc = ctypes.CDLL(None)
address = lambda f: ctypes.cast(f, ctypes.c_void_p).value
class Kernel:
    pass
slow = type(scale._plan)(address(libc.usleep), address(libc.abs), 0, 300000)
args = (x, 2.0)
assert not slow.repeats(args) and slow.repeats(args)
# (another thread's call in between: its arguments are not recorded with this one's results)
assert not slow.repeats((x[:1], 2.0)) and slow.record(args, [1], [x], [2], False, 0)
assert slow.call(Kernel(), args, lambda device: 0) is None and slow.call(Kernel(), (x[:1], 2.0), lambda device: 0) is None
assert not slow.repeats(args) and slow.repeats(args) and slow.record(args, [1], [x], [2], False, 0)
before = beats[0]
time.sleep(0.3)
free = beats[0] - before
before = beats[0]
assert slow.call(Kernel(), args, lambda device: 0).shape == x.shape
ran = beats[0] - before
stop.set(); t.join()
assert ran > free / 3, (ran, free)

# the same kernels from several threads, a stream each: every call reads and writes its own tensors
failed = []
def work(n):
    try:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(stream):
            for i in range(200):
                y = x + float(n * 1000 + i)
                got = scale(y, 2.0)
                c = product(a, b) if i % 8 == 0 else None
                stream.synchronize()
                if not torch.equal(got, y * 2.0):
                    failed.append((n, i))
                if c is not None and not torch.equal(c.double(), want):
                    failed.append((n, i, "product"))
    except Exception as e:
        failed.append(repr(e))
threads = [threading.Thread(target=work, args=(n,)) for n in range(4)]
[w.start() for w in threads]
[w.join(90) for w in threads]
assert not any(w.is_alive() for w in threads)
assert not failed, failed[:5]

# shapes and numbers of their own: some calls come from the plan, some from Python
failed = []
def mixed(n):
    try:
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(stream):
            for i in range(200):
                y = x[: 1 + (n + i // 5) % 3 * 20] + float(i)
                f = 2.0 if i % 3 else float(n)
                got = scale(y, f)
                stream.synchronize()
                if got.shape != y.shape or not torch.equal(got, y * f):
                    failed.append((n, i))
    except Exception as e:
        failed.append(repr(e))
threads = [threading.Thread(target=mixed, args=(n,)) for n in range(4)]
[w.start() for w in threads]
[w.join(90) for w in threads]
assert not any(w.is_alive() for w in threads) and not failed, failed[:5]
print("threads: ok")
'''


def test_several_threads_call_the_same_kernel():
    _run(_THREADS, "threads: ok")


def _run(script, said):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root + os.pathsep + os.environ.get("PYTHONPATH", ""))
    r = subprocess.run([sys.executable, "-c", script], cwd=root, env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and said in r.stdout, r.stdout + r.stderr


def test_what_changes_the_kernel_between_two_calls():
    _run(_CHANGES, "changes: ok")


def test_plans():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root + os.pathsep + os.environ.get("PYTHONPATH", ""))
    r = subprocess.run([sys.executable, "-c", _SCRIPT], cwd=root, env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and "plans: ok" in r.stdout, r.stdout + r.stderr
