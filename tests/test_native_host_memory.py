"""The native host code where memory runs out: an exception of C++ must not leave a function that the interpreter
calls (it would end the process), and what the fast path cannot do is left to the Python code."""
import os
import subprocess
import sys

from quantfour_adamw_cuda_amd import build as q4build

HERE = os.path.dirname(os.path.abspath(__file__))

# no GPU: a plan over no parameters, with state objects to hold, goes through every allocation but the buckets' own
EVERY_ALLOCATION = r"""
import ctypes, importlib.util, sys
import torch
spec = importlib.util.spec_from_file_location("_q4host", sys.argv[1])
h = importlib.util.module_from_spec(spec)
spec.loader.exec_module(h)
fail_after = ctypes.CDLL(sys.argv[1]).fail_after
fail_after.argtypes = [ctypes.c_long]
d, t = {"step": 1}, torch.zeros(0)
args = ((), t, [(d, 1, 2, 3)] * 3, [(d, "k", 4)] * 5, [])
whole = 0
for n in range(64):
    fail_after(n)
    plan = h.plan(*args)
    fail_after(-1)
    if plan is None:
        continue
    whole += 1
    del plan
    if whole == 2:
        break
assert whole == 2 and n > 3, (whole, n)     # some allocations failed, and with enough of them the plan is made
assert h.plan(*args) is not None
print("memory: ok")
"""


def test_no_allocation_failure_leaves_the_module(tmp_path):
    out = str(tmp_path / "_q4host.so")
    q4build.compile_host_module(out, extra=["-Wl,-Bsymbolic", os.path.join(HERE, "native", "failing_new.cpp")])
    run = subprocess.run([sys.executable, "-c", EVERY_ALLOCATION, out], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert run.returncode == 0 and "memory: ok" in run.stdout, run.stdout[-3000:]
