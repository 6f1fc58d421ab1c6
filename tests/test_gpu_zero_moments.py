"""Zeros in the exact parameter update, which take neither the short sequences nor the general
expansions, and tiles whose moments are all zero, which store their codes and scales only where
they are not in place; NaN moments of any payload, which get code 0 from the fixed-point codes."""
import numpy as np
import pytest
import torch

import quantfour_adamw_cuda_amd as q4
from oracle import q4_oracle as oc
from oracle import q4_oracle_torch as ot
from tests.q4_testlib import HP, DeviceTensor, OracleTensor, assert_state_equal, bits

pytestmark = pytest.mark.gpu


def _pair(n, gen, cuda):
    p = torch.randn(n, generator=gen) * 0.02
    p[::7] = 0.0
    p[3::7] = -0.0
    dev = DeviceTensor(p, cuda)
    return dev, OracleTensor(p)


def _set_state(dev, ref, m, v, sm, sv):
    for name, x in (("m", m), ("v", v), ("sm", sm), ("sv", sv)):
        getattr(dev, name).copy_(x)
        getattr(ref, name)[:] = x.numpy()


def _step(dev, ref, g, cuda, step, what):
    q4.fused_4bit(dev.p, g.to(cuda), dev.m, dev.v, dev.sm, dev.sv, HP["beta1"], HP["beta2"], HP["lr"], HP["weight_decay"], HP["eps"], step)
    prev = ref.step(g, step)
    assert_state_equal(dev, ref, prev, what)
    # signs of zeros too (a NaN's bits are the machine's)
    got = dev.p.cpu().numpy()
    num = ~np.isnan(ref.p)
    assert np.array_equal(bits(got)[num], bits(ref.p)[num]) and np.isnan(got[~num]).all(), what


@pytest.mark.parametrize("n", [128, 256, 1024, 4096 + 256, 4096 + 37])
@pytest.mark.parametrize("state", ["fresh", "stale codes", "negative zeros", "in training"])
def test_zero_gradients(cuda, n, state):
    """whole tensors, tiles, blocks and single elements of zeros of either sign"""
    gen = torch.Generator().manual_seed(n)
    dev, ref = _pair(n, gen, cuda)
    nbytes, nblk = oc.state_sizes(n)
    if state != "fresh":
        m = torch.randint(0, 256, (nbytes,), dtype=torch.uint8, generator=gen)
        v = torch.randint(0, 256, (nbytes,), dtype=torch.uint8, generator=gen)
        if n % 2:
            m[-1] &= 15
            v[-1] &= 15
        sm, sv = torch.zeros(nblk), torch.zeros(nblk)
        if state == "negative zeros":
            sm[:] = -0.0
        if state == "in training":
            sm[:] = torch.rand(nblk, generator=gen) * 1e-3
            sv[:] = torch.rand(nblk, generator=gen) * 1e-6
        _set_state(dev, ref, m, v, sm, sv)
    for step, share in enumerate((1.0, 0.5, 0.9, 1.0), 1):
        g = torch.randn(n, generator=gen) * 1e-3
        g[torch.rand(n, generator=gen) < share] = 0.0
        g[torch.rand(n, generator=gen) < 0.3] *= -0.0
        if share < 1.0 and n > 512:
            g[256:512] = 0.0
        _step(dev, ref, g, cuda, step, f"{state}, step {step}")


@pytest.mark.parametrize("value", [1e-38, 1e-30, 1e-20, 1e-19, 1e10, 1e15, 1e25])
def test_zeros_beside_moments_out_of_range(cuda, value):
    """a lane with zeros and one value that only the general expansions cover"""
    n = 1024
    gen = torch.Generator().manual_seed(5)
    dev, ref = _pair(n, gen, cuda)
    for step in (1, 2):
        g = torch.zeros(n)
        g[torch.randint(0, n, (40,), generator=gen)] = value
        g[torch.randint(0, n, (40,), generator=gen)] = -0.01
        _step(dev, ref, g, cuda, step, f"{value}, step {step}")


@pytest.mark.parametrize("pattern", [0x7FC00000, 0x7FC00123, 0x7FD48001, 0x7FFFFFFF, 0xFFC0FFFF - (1 << 32), 0xFFFFFFFF - (1 << 32)])
@pytest.mark.parametrize("grads", ["float32", "bfloat16"])
def test_nan_payloads(cuda, pattern, grads):
    n = 1024
    gen = torch.Generator().manual_seed(9)
    dev, ref = _pair(n, gen, cuda)
    g = torch.randn(n, generator=gen) * 1e-3
    at = torch.randint(0, n, (30,), generator=gen)
    g[at] = torch.full((30,), pattern, dtype=torch.int32).view(torch.float32)
    g[256:384] = torch.full((128,), pattern, dtype=torch.int32).view(torch.float32)
    if grads == "bfloat16":
        g = g.to(torch.bfloat16)
    q4.fused_4bit(dev.p, g.to(cuda), dev.m, dev.v, dev.sm, dev.sv, HP["beta1"], HP["beta2"], HP["lr"], HP["weight_decay"], HP["eps"], 1)
    ref.step(g.float(), 1)
    assert np.array_equal(dev.m.cpu().numpy(), ref.m) and np.array_equal(dev.v.cpu().numpy(), ref.v)
    assert np.array_equal(bits(dev.sm.cpu().numpy()), bits(ref.sm)) and np.array_equal(bits(dev.sv.cpu().numpy()), bits(ref.sv))


@pytest.mark.parametrize("value", [1e-44, 1e-38, 1e-25, 1e-20, 1e18, 1e19])
@pytest.mark.parametrize("zeros", [0.0, 0.1])
def test_moments_out_of_range(cuda, value, zeros):
    """lanes all of whose moments lie outside the short sequences' ranges, with and without zeros among them"""
    n = 4096 + 37
    gen = torch.Generator().manual_seed(6)
    dev, ref = _pair(n, gen, cuda)
    for step in (1, 2, 3):
        g = (torch.rand(n, generator=gen) + 0.5) * value * torch.sign(torch.randn(n, generator=gen))
        g[torch.rand(n, generator=gen) < zeros] = 0.0
        _step(dev, ref, g, cuda, step, f"{value}, step {step}")


# every payload whose upper half is all ones reaches the noise's addition at the top of the 32-bit range
ONES = {"float32": (torch.int32, torch.float32, [0xFFFFFFFF, 0xFFFF8001, 0x7FFFFFFF, 0xFFC00001]),
        "bfloat16": (torch.int16, torch.bfloat16, [0xFFFF]), "float16": (torch.int16, torch.float16, [0xFFFF, 0x7FFF])}


@pytest.mark.parametrize("rank1", [False, True])
@pytest.mark.parametrize("p_dt", ["float32", "float16"])
@pytest.mark.parametrize("g_dt,pattern", [(k, x) for k, v in ONES.items() for x in v[2]])
def test_nan_payloads_stochastic(cuda, g_dt, pattern, p_dt, rank1):
    """stochastic rounding: code 0 for a NaN moment, single elements, half a row and whole blocks of them"""
    ints, dt, _ = ONES[g_dt]
    rows, cols, seed = 96, 768, 0x1234_5678_9ABC
    gen = torch.Generator().manual_seed(pattern & 0xFFFF)
    p = (torch.randn(rows, cols, generator=gen) * 0.02).to(getattr(torch, p_dt))
    g = (torch.randn(rows, cols, generator=gen) * 1e-3).to(dt)
    bits_ = g.view(ints)
    value = pattern - (1 << (32 if ints is torch.int32 else 16)) if pattern >> (31 if ints is torch.int32 else 15) else pattern
    bits_[torch.rand(rows, cols, generator=gen) < 0.02] = value
    bits_[5, :384] = value
    bits_[40:42] = value
    n = rows * cols
    zeros = lambda k, d=torch.float32: torch.zeros(k, dtype=d)
    nbytes, nblk = oc.state_sizes(n)
    m, v, sm = zeros(nbytes, torch.uint8), zeros(nbytes, torch.uint8), zeros(nblk)
    hpa = (HP["beta1"], HP["beta2"], HP["lr"], HP["weight_decay"], HP["eps"], 1)
    g32 = torch.where(torch.isnan(g.float()), torch.nan, g.float())
    with np.errstate(invalid="ignore"):
        if rank1:
            want = ot.step_quant_rank1_sr(p, g32, m, v, sm, zeros(rows), zeros(cols), step=1, seed=seed, tensor_salt=0, **HP)[1:]
        else:
            want = ot.step_quant_sr(p.view(-1), g32.view(-1), m, v, sm, zeros(nblk), step=1, seed=seed, tensor_salt=0, **HP)[1:]
    d = lambda t: t.clone().to(cuda)
    if rank1:
        got = [d(m), d(v), d(sm), d(zeros(rows)), d(zeros(cols))]
        q4.quantfour_hip.fused_4bit_rank1_multi([d(p)], [d(g)], *[[t] for t in got], [d(zeros(rows))], [d(zeros(cols))], *hpa, seed=seed)
    else:
        got = [d(m), d(v), d(sm), d(zeros(nblk))]
        q4.quantfour_hip.fused_4bit_multi_sr([d(p).view(-1)], [d(g).view(-1)], *[[t] for t in got], *hpa, seed)
    names = ("m codes", "v codes", "m scales", "v scales or rows", "columns")
    for name, a, b in zip(names, got, want):
        a, b = a.cpu(), b.reshape(-1)
        if a.dtype == torch.float32:
            a, b = a.view(torch.int32), b.contiguous().view(torch.int32)
        bad = torch.nonzero(a != b).reshape(-1)
        assert bad.numel() == 0, f"{name}: {bad.numel()} differ, first {bad[:4].tolist()}: {a[bad[:4]].tolist()} for {b[bad[:4]].tolist()}"
