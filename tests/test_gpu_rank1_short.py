"""Rank-1 scaling of tensors with several leading dimensions: cancelled steps of the kernel for short rows and of the leading
statistics, lists around the number of short-row tensors that a launch's arguments hold (25), and the leading
statistics' larger tiles."""
import pytest
import torch

from oracle import q4_oracle_torch as ot
from quantfour_adamw_cuda_amd import quantfour_hip as q
from tests import test_gpu_rank1 as base
from tests.q4_testlib import HP, grads_config1

pytestmark = pytest.mark.gpu


class _Tensor:
    def __init__(self, p, device):
        n, cols = p.numel(), p.shape[-1]
        z = lambda m, dt=torch.float32: torch.zeros(m, dtype=dt, device=device)
        self.p = p.clone().to(device)
        self.m, self.v, self.sm = z((n + 1) // 2, torch.uint8), z((n + 1) // 2, torch.uint8), z((n + 127) // 128)
        self.r, self.c, self.rn, self.cn = z(n // cols), z(cols), z(n // cols), z(cols)
        self.lead = ([z(d) for d in p.shape[:-1]], [z(d) for d in p.shape[:-1]]) if p.dim() > 2 else None

    def state(self):
        return [self.p, self.m, self.v, self.sm, self.r, self.c, *(self.lead[0] if self.lead else [])]

    def scratch(self):
        return [self.rn, self.cn, *(self.lead[1] if self.lead else [])]


def _step(ts, gs, step, **kw):
    pick = lambda k: [getattr(t, k) for t in ts]
    q.fused_4bit_rank1_multi(pick("p"), gs, pick("m"), pick("v"), pick("sm"), pick("r"), pick("c"), pick("rn"), pick("cn"), *base.HPA, step,
                             leads=pick("lead"), **kw)


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("shape", [(5, 40, 3, 3), (6, 70, 1, 5), (33, 7, 5),
                                   (4, 30, 96), (3, 20, 264),       # scales from vectors; leading statistics of the wide form
                                   (2, 3073, 128)])                 # several runs in a workgroup of the leading statistics
def test_cancelled_steps_leave_everything(cuda, shape, p_dt, g_dt):
    """An overflow flag after a step: parameters, codes, statistics and the rows' scales, which the kernel for short rows
    writes itself, stay; the gradients are cleared only where that is asked for."""
    gen = torch.Generator().manual_seed(sum(shape))
    t = _Tensor((torch.randn(shape, generator=gen) * 0.05).to(base.DT[p_dt]), cuda)
    g = grads_config1(gen, t.p.numel()).view(shape).to(base.DT[g_dt]).to(cuda)
    _step([t], [g], 1)
    before, g0 = [x.clone() for x in t.state()], (g * 8).clone()
    g.mul_(8)                                                       # other maxima than the ones that are there
    flag = torch.ones(1, device=cuda)
    for kw in ({}, dict(zero_grad=True)):
        _step([t], [g], 2, found_inf=flag, **kw)
        for a, b in zip(before, t.state()):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), f"{shape} {kw}"
        assert not any(bool(x.any()) for x in t.scratch()), f"{shape} {kw}: scratch"
        assert torch.equal(g, torch.zeros_like(g) if kw else g0), f"{shape} {kw}: gradients"
    _step([t], [g0], 2, found_inf=torch.zeros(1, device=cuda))      # and the step is still there to be taken
    assert not torch.equal(before[3], t.sm) and not torch.equal(before[4], t.r)


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("others", [0, 3, 8])
@pytest.mark.parametrize("count", [24, 25, 26, 51])
def test_lists_of_short_rows(cuda, count, others, p_dt, g_dt):
    """Lists that end just before, at and after the 25 short-row tensors of a launch, alone and with tensors of other
    kernels before them and after them (with 8, the batch's 32 tensors are met too): every tensor steps once, as it does by itself."""
    more = [(66, 1024), (40, 64), (30, 301), (20, 520), (3, 5, 64), (33, 77), (2, 9, 264), (4100, 3)]
    short = [(2 + i % 5, 3 + i % 7, 3, 3) if i % 3 else (4 + i % 4, 30 + i, 5) for i in range(count)]
    shapes = more[:others // 2] + short + more[others // 2:others]
    gen = torch.Generator().manual_seed(count * 100 + others)
    ps = [(torch.randn(s, generator=gen) * 0.05).to(base.DT[p_dt]) for s in shapes]
    together, alone = [_Tensor(p, cuda) for p in ps], [_Tensor(p, cuda) for p in ps]
    for step in (1, 2):
        gs = [grads_config1(gen, p.numel()).view(p.shape).to(base.DT[g_dt]).to(cuda) for p in ps]
        _step(together, gs, step)
        for i, t in enumerate(alone):
            _step([t], [gs[i]], step)
            for a, b in zip(t.state(), together[i].state()):
                assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), f"step {step}: tensor {i} {shapes[i]}"
            assert not any(bool(x.any()) for x in together[i].scratch()), f"step {step}: tensor {i} {shapes[i]}: scratch"


# A workgroup takes 32 indices of the first dimension, doubled up to 256 while 768 workgroups of that many indices and of
# 256 (fp32 gradients) or 512 elements below them are left: 128 from 768 * 128 * 256 = 25.2 million elements on, 256 from 50.4
# million, twice as many with 16-bit gradients.
@pytest.mark.parametrize("shape,g_dt,taken", [((300, 9400, 3, 3), torch.float32, 128),        # the last workgroup has 44
                                              ((400, 14100, 3, 3), torch.float32, 256),       # 144
                                              ((257, 65500, 6), torch.bfloat16, 256)])        # 1
def test_statistics_of_larger_tiles(cuda, shape, g_dt, taken):
    n, cols = 1, shape[-1]
    for d in shape:
        n *= d
    run = 256 if g_dt == torch.float32 else 512
    assert n // (run * taken) >= 768 and (taken == 256 or n // (run * taken * 2) < 768)
    gen = torch.Generator(device=cuda).manual_seed(taken)
    t = _Tensor(torch.randn(shape, generator=gen, device=cuda) * 0.05, cuda)
    stat = lambda j: torch.zeros([d if i == j else 1 for i, d in enumerate(shape)], device=cuda)
    ref = (t.p.clone(), t.m.clone(), t.v.clone(), t.sm.clone(), [stat(j) for j in range(len(shape))])
    weight = torch.rand([shape[0]] + [1] * (len(shape) - 1), generator=gen, device=cuda)
    for step in (1, 2):
        g = (torch.randn(shape, generator=gen, device=cuda) * weight).to(g_dt)
        with torch.no_grad():
            ref = ot.step_quant_rank1_nd(ref[0], g, *ref[1:], step=step, **HP)
        _step([t], [g], step)
        for j, (have, want) in enumerate(zip(t.lead[0] + [t.c], ref[4])):
            assert torch.equal(have, want.reshape(-1)), f"step {step}: statistic {j}"
        assert torch.equal(t.m, ref[1]) and torch.equal(t.v, ref[2]), f"step {step}: codes"
