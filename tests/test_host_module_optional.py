"""The package without its native host module: the module makes steps' host part faster and does nothing that the
Python code does not, so a missing one costs speed and nothing else."""
import os
import shutil
import subprocess
import sys

import pytest
import torch

import quantfour_adamw_cuda_amd as package
from quantfour_adamw_cuda_amd import AdamWFused_QuantFour, _lib
from quantfour_adamw_cuda_amd import quantfour_hip as q

HP = (0.9, 0.999, 1e-3, 0.01, 1e-8)

WITHOUT = r"""
import warnings
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    import torch
    from quantfour_adamw_cuda_amd import AdamWFused_QuantFour, _lib, fused_4bit, state_sizes
    L = _lib.load()
    _lib.load()
assert L.q4adamw_version() >= 1000 and state_sizes(129) == (65, 2)
assert len([w for w in seen if "_q4host" in str(w.message)]) == 1, [str(w.message) for w in seen]
z = torch.zeros
try:
    fused_4bit(z(200), z(200), z(100, dtype=torch.uint8), z(100, dtype=torch.uint8), z(2), z(2), 0.9, 0.999, 1e-3, 0.01, 1e-8, 1)
except AssertionError as e:
    assert "param must be on cuda" in str(e)      # the Python code's own refusal
else:
    raise SystemExit("taken")
p = torch.nn.Parameter(z(5000))
p.grad = z(5000)
try:
    AdamWFused_QuantFour([p]).step(max_grad_norm=1.0)
except (AssertionError, RuntimeError) as e:
    assert "_q4host" not in str(e), e
print("without: ok")
"""


def test_the_package_works_without_the_module(tmp_path):
    src = os.path.dirname(package.__file__)
    shutil.copytree(src, tmp_path / "quantfour_adamw_cuda_amd", ignore=shutil.ignore_patterns("_q4host*", "__pycache__"))
    out = subprocess.run([sys.executable, "-c", WITHOUT], cwd=tmp_path, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                         timeout=300, env=dict(os.environ, PYTHONPATH=str(tmp_path)))
    assert out.returncode == 0 and "without: ok" in out.stdout, out.stdout[-3000:]


@pytest.mark.parametrize("tag,version", [(None, None), ("torch 2.0.0 0 cpython-310", 0), ("torch 2.0.0 0 cpython-310", None), (None, 0)])
def test_a_module_of_another_build_is_not_used(monkeypatch, tag, version):
    """A module that reads tensors as another torch lays them out, or calls the library as another version declares it,
    is never handed the library's entry points."""
    L = _lib.load()
    other = type("other", (), {"bind": staticmethod(lambda *a: pytest.fail("bound"))})
    if tag is not None or version is not None:        # without either: a module that says nothing of its build
        other.built_for = tag or _lib.host_module_tag()
        other.library_version = L.q4adamw_version() + (1 if version is not None else 0)
    monkeypatch.setattr(package, "_q4host", other, raising=False)
    monkeypatch.setitem(sys.modules, "quantfour_adamw_cuda_amd._q4host", other)
    with pytest.warns(UserWarning, match="_q4host was built for"):
        assert _lib._bind_host(L) is _lib.PythonHost


def test_the_built_module_is_used():
    L = _lib.load()
    assert _lib.host.built_for == _lib.host_module_tag() and _lib.host.library_version == L.q4adamw_version()
    assert _lib.host.built_for.startswith("torch " + torch.__version__)


@pytest.mark.gpu
@pytest.mark.parametrize("p_dt,g_dt", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
def test_results_without_the_module(cuda, monkeypatch, p_dt, g_dt):
    """Steps, a clipped one among them, and direct calls with and without it: the same bits."""
    gen = torch.Generator(device=cuda).manual_seed(11)
    base = [(torch.randn(s, generator=gen, device=cuda) * 0.05).to(p_dt) for s in ((70, 129), (100,), (64, 512))]
    grads = [[(torch.randn(b.shape, generator=gen, device=cuda) * 1e-2).to(g_dt) for b in base] for _ in range(3)]
    with_module = _lib.load() and _lib.host

    def run():
        ps = [torch.nn.Parameter(b.clone()) for b in base]
        opt = AdamWFused_QuantFour(ps, lr=1e-3)
        for k, gs in enumerate(grads):
            for p, g in zip(ps, gs):
                p.grad = g.clone()
            opt.step(**(dict(max_grad_norm=0.5) if k == 1 else {}))
        n = base[0].numel()
        nb, nk = q.state_sizes(n)
        z = lambda m, dt=torch.float32: torch.zeros(m, dtype=dt, device=cuda)
        direct = [base[0].clone(), z(nb, torch.uint8), z(nb, torch.uint8), z(nk), z(nk)]
        small = [base[1].clone(), z(100), z(100)]
        q.fused_4bit(direct[0], grads[0][0], *direct[1:], *HP, 1)
        q.fused_single_tensor(small[0], grads[0][1], *small[1:], *HP, 1)
        return [p.detach() for p in ps] + direct + small, opt._plans[0].native is not None

    fast, native = run()
    assert native, "the built module is not in use"
    monkeypatch.setattr(_lib, "host", _lib.PythonHost)
    plain, native = run()
    assert not native and _lib.host is not with_module
    for a, b in zip(fast, plain):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
