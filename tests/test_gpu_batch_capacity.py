"""Tensor lists around the number of descriptors a launch's arguments hold (61 quantized, 103
small), with every tensor's last chunk of another length: each tensor steps exactly once."""
import numpy as np
import pytest
import torch

import quantfour_adamw_cuda_amd as q4
from oracle import q4_oracle as oc
from tests.q4_testlib import HP, DeviceTensor, OracleTensor, assert_state_equal, bits, grads_config1

pytestmark = pytest.mark.gpu
HPA = (HP["beta1"], HP["beta2"], HP["lr"], HP["weight_decay"], HP["eps"])


@pytest.mark.parametrize("count", [1, 7, 8, 60, 61, 62, 123])
def test_quantized(cuda, count):
    gen = torch.Generator().manual_seed(count)
    sizes = [int(torch.randint(1, 3000, (1,), generator=gen)) for _ in range(count)]
    devs = [DeviceTensor(torch.randn(n, generator=gen) * 0.02, cuda) for n in sizes]
    refs = [OracleTensor(d.p.cpu()) for d in devs]
    gs = [grads_config1(gen, n) for n in sizes]
    q4.fused_4bit_multi([d.p for d in devs], [g.to(cuda) for g in gs], [d.m for d in devs], [d.v for d in devs],
                        [d.sm for d in devs], [d.sv for d in devs], *HPA, 1)
    for i, (d, r, g) in enumerate(zip(devs, refs, gs)):
        assert_state_equal(d, r, r.step(g, 1), f"tensor {i} of {count}")


@pytest.mark.parametrize("count", [1, 7, 8, 15, 102, 103, 104, 207])
def test_small(cuda, count):
    gen = torch.Generator().manual_seed(count)
    sizes = [(1, 1023, 1024, 1025, 2048, 4096, 77)[i % 7] if i % 3 else int(torch.randint(1, 5000, (1,), generator=gen)) for i in range(count)]
    ps = [torch.randn(n, generator=gen) * 0.02 for n in sizes]
    gs = [grads_config1(gen, n) for n in sizes]
    dp = [p.to(cuda) for p in ps]
    dm, dv = [torch.zeros_like(p) for p in dp], [torch.zeros_like(p) for p in dp]
    q4.fused_single_tensor_multi(dp, [g.to(cuda) for g in gs], dm, dv, *HPA, 1)
    for i in range(count):
        p, m, v = ps[i].numpy().copy(), np.zeros(sizes[i], np.float32), np.zeros(sizes[i], np.float32)
        oc.step_unquant(p, gs[i].numpy(), m, v, step=1, **HP)
        for got, want, what in ((dp[i], p, "p"), (dm[i], m, "m"), (dv[i], v, "v")):
            assert np.array_equal(bits(got.cpu().numpy()), bits(want)), f"tensor {i} of {count} ({sizes[i]}): {what}"
