"""The native host code under UndefinedBehaviorSanitizer, and where memory runs out: an exception of C++ must not leave
a function that the interpreter calls (it would end the process), and what the fast path cannot do is left to the Python
code."""
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
d, t = {"step": 1, "exp_avg": 2, "exp_avg_sq": 3, "k": 4}, torch.zeros(0)
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
plan = h.plan(*args)
# what a process without a GPU reaches of the rest
assert h.refresh(plan, [], t) is True and h.refresh(plan, [t], t) is False and h.refresh(plan, [], torch.zeros(0)) is False
d["step"] = 5
assert h.refresh(plan, [], t) is False
hyper = (0.9, 0.999, 1e-3, 0, 1e-8)
assert h.run(plan, *hyper, 0, 7) is None and h.run(plan, *hyper[:4], "1e-8", 0, 7) is None and h.run(plan, *hyper[:4], 10 ** 400, 0, 7) is None
p, codes = torch.zeros(200), torch.zeros(100, dtype=torch.uint8)
assert h.fused_4bit(p, p, codes, codes, p[:2], p[:2], *hyper, 1) is None and h.fused_single_tensor(p, p, p, p, *hyper, 1) is None
par = torch.nn.Parameter(p)
table = (ctypes.c_uint64 * 4)()
assert h.gradients(([par, par],), ctypes.addressof(table), 2) is None      # without gradients
par.grad = p
assert h.gradients(([par], [par]), ctypes.addressof(table), 1) is None and h.gradients(([None],), ctypes.addressof(table), 2) is None
for bad in ((1,), (par, t, [], [], []), ((par,), t, [], [], []), ((), t, [1], [], []), ((), t, [], [(d, "k")], []), ((), p, [], [], [])):
    assert h.plan(*bad) is None
try:
    h.plan((), t, [], [], [(1, [0], 0, 0, 0, 0, 0)])
except ValueError as e:
    assert "index" in str(e)
else:
    raise SystemExit("an index past the parameters was taken")
print("memory: ok")
"""


def test_host_module_under_sanitizer_and_without_memory(tmp_path):
    out = str(tmp_path / "_q4host.so")
    q4build.compile_host_module(out, extra=["-fsanitize=undefined", "-fno-sanitize=vptr", "-fno-sanitize-recover=undefined", "-Wl,-Bsymbolic", os.path.join(HERE, "native", "failing_new.cpp")])
    run = subprocess.run([sys.executable, "-c", EVERY_ALLOCATION, out], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert run.returncode == 0 and "memory: ok" in run.stdout, run.stdout[-3000:]
