"""Every chunk of a grid is taken exactly once, whatever the length of the runs of chunks that go
to one XCD: grids around powers of two, where the run length doubles from 512 << k on (up to runs of 64,
from 2^19 chunks on of 1024), and grids with a remainder beyond whole rounds of runs.  A chunk taken twice would step twice, one left
out not at all."""
import pytest
import torch

from tests.q4_testlib import DeviceTensor, OracleTensor, HP, assert_state_equal, grads_config1
import quantfour_adamw_cuda_amd as q4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 128, 255, 256, 511, 513, 1023, 1024, 2047, 2048, 2049, 2560, 3071])
def test_grid_sizes(cuda, chunks):
    n = chunks * 1024 - (37 if chunks % 2 else 0)
    gen = torch.Generator().manual_seed(chunks)
    dev = DeviceTensor(torch.randn(n, generator=gen) * 0.02, cuda)
    ref = OracleTensor(dev.p.cpu())
    g = grads_config1(gen, n)
    q4.fused_4bit(dev.p, g.to(cuda), dev.m, dev.v, dev.sm, dev.sv, HP["beta1"], HP["beta2"], HP["lr"], HP["weight_decay"], HP["eps"], 1)
    prev = ref.step(g, 1)
    assert_state_equal(dev, ref, prev, f"{chunks} chunks")
