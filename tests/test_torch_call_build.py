"""The extension behind repeated calls on torch tensors, where it cannot be used: garbage in its place, or built for another torch.
Calls then stay in Python, and nothing raises. In a process of its own that imports torch first (see tests/test_torch_adapter.py
for why); no GPU is needed."""
import os
import subprocess
import sys

import pytest

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_SCRIPT = r'''
import os, sys
import torch
from dvm_amd import _core, build
case, tmp = sys.argv[1:]
if case == "garbage":
    with open(os.path.join(tmp, "_torch_call.so"), "wb") as f:
        f.write(b"not a library")
if case in ("garbage", "missing"):
    address = _core._lib.dvm_rt_plan_stamp  # (libdvm.so is loaded from where it is)
    _core._LIB_DIR = tmp
if case == "other torch":
    torch.__version__ = "0.1"
for _ in range(3):
    plan = _core.new_call_plan(0)
    assert (plan is not None) == (case == "as built"), case
if case == "as built":
    assert _core._call_module().built_for == build.torch_call_tag()
print("ok")
'''


@pytest.mark.parametrize("case", ["as built", "garbage", "missing", "other torch"])
def test_an_extension_that_cannot_be_used_is_left_alone(case, tmp_path):
    if case != "garbage" and case != "missing" and not os.path.exists(os.path.join(_ROOT, "dvm_amd", "lib", "_torch_call.so")):
        pytest.skip("the extension has not been built")
    env = dict(os.environ, PYTHONPATH=_ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""))
    r = subprocess.run([sys.executable, "-c", _SCRIPT, case, str(tmp_path)], cwd=_ROOT, env=env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
    assert ("stay in Python" in r.stderr) == (case in ("garbage", "other torch")), r.stderr


_STALE = r'''
import os, sys
from dvm_amd import build
if build.torch_call_tag() is None:
    sys.exit("no torch")
build.LIB = build.OBJ = sys.argv[1]
library = os.path.join(sys.argv[1], "_torch_call.so")

def compiled():  # whether a build would compile it; a stand-in for the library is left as a compiler would leave one
    command = build.torch_call_job()
    assert command is None or not os.path.exists(library)
    if command is not None:
        open(library, "wb").close()
    return command is not None

assert compiled() and not compiled() and not compiled()
build.torch_call_tag = lambda: "torch 0.1, cpython-0"
assert compiled() and not compiled()
os.remove(library)
assert '-DDVM_TORCH_CALL_TAG="torch 0.1, cpython-0"' in build.torch_call_job()
print("ok")
'''


def test_what_the_extension_is_compiled_for_decides_whether_it_is_out_of_date(tmp_path):
    r = subprocess.run([sys.executable, "-c", _STALE, str(tmp_path)], cwd=_ROOT, env=dict(os.environ, PYTHONPATH=_ROOT), capture_output=True, text=True, timeout=300)
    if "no torch" in r.stderr:
        pytest.skip("no torch, or no headers of the interpreter")
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
