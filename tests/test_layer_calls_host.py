"""Host code of the layer calls on host arrays, run without a GPU on a stand-in
for the HIP calls they make (native/hip_stub.c): how they allocate, and what they
report when a launch fails."""
import os
import shutil
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc missing")

CHILD = """
import sys
import numpy as np
sys.path.insert(0, %r)
from conftest import load_pkg
P = load_pkg()
call, grid, batch = sys.argv[1], tuple(int(v) for v in sys.argv[2].split("x")), int(sys.argv[3])
x = np.zeros((batch, grid[0] * grid[1] * grid[2], 32), np.float32)
w = np.zeros((27, 32, 32), np.float32)
try:
    P.conv_forward(grid, x, w) if call == "forward" else P.conv_backward(grid, x, w, x)
    print("ok")
except P.PlsqrError as e:
    print("error", e.code, str(e))
""" % os.path.join(ROOT, "tests")


def layer_call(tmp_path, call, grid, batch=1, launch=0):
    """The child's last line and the sizes it allocated."""
    stub = str(tmp_path / "hip_stub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", stub, os.path.join(ROOT, "tests", "native", "hip_stub.c")],
                   check=True)
    env = dict(os.environ, HIP_STUB_LAUNCH=str(launch))
    env["LD_PRELOAD"] = " ".join([stub, env.get("LD_PRELOAD", "")]).strip()
    r = subprocess.run([sys.executable, "-c", CHILD, call, grid, str(batch)], capture_output=True, text=True, timeout=300,
                       env=env)
    assert r.returncode == 0, r.stderr[-3000:]
    lines = r.stdout.splitlines()
    return lines[-1], [int(l.split()[1]) for l in lines if l.startswith("alloc ")]


@pytest.mark.parametrize("call,grid,most", [("forward", "8x8x128", 2), ("forward", "3x3x3", 1), ("backward", "8x8x64", 2),
                                            ("forward", "32x32x32", 1), ("backward", "31x27x35", 1)])
def test_small_buffers_stay_on_the_fast_allocations(tmp_path, call, grid, most):
    """An hipMalloc of 2 MiB or more costs several smaller ones: up to 4 MiB in
    all are spread over allocations below it, more are one."""
    last, sizes = layer_call(tmp_path, call, grid)
    assert last == "ok" and 1 <= len(sizes) <= most
    if sum(sizes) <= 4 << 20:
        assert max(sizes) < 2 << 20
    else:
        assert len(sizes) == 1


@pytest.mark.parametrize("call", ["forward", "backward"])
def test_a_failed_launch_is_reported_with_its_message(tmp_path, call):
    last, _ = layer_call(tmp_path, call, "5x4x3", launch=1)
    assert last.startswith("error 4 plsqr error HIP: ") and last != "error 4 plsqr error HIP: ", last
