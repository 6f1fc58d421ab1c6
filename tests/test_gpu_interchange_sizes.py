"""Checkpoint quantize / dequantize where their tiles end: a workgroup takes 2048 elements to encode and
4096 to decode, a wave two and four tiles of 256, a lane four elements of each; code buffers at odd
addresses; matrices whose rows end inside a lane's four elements."""
import numpy as np
import pytest
import torch

from oracle import q4_oracle as oc
from oracle import q4_oracle_torch as ot
from quantfour_adamw_cuda_amd import _lib
from quantfour_adamw_cuda_amd import quantfour_hip as q
from tests.q4_testlib import bits, grads_config1

pytestmark = pytest.mark.gpu


def _values(gen, n, which):
    """scales from 1e-38 to 1e36 (in and out of the reciprocal's range), zeros, NaN, infinity, both signs"""
    x = grads_config1(gen, n) * torch.pow(10.0, torch.randint(-35, 37, ((n + 127) // 128,), generator=gen).float()).repeat_interleave(128)[:n]
    if n > 400:
        x[130:133] = float("nan")
        x[300] = float("inf")
        x[256:280] = 0.0
    return x * x if which and n % 2 else x


@pytest.mark.parametrize("n", [3, 4, 253, 255, 257, 1023, 1025, 4095, 4096, 4097, 12290, 100001])
@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("odd", [0, 1])
def test_blocks(cuda, n, which, odd):
    x = _values(torch.Generator().manual_seed(n * 2 + which), n, which)
    L, nbytes, nblk = _lib.load(), (n + 1) // 2, (n + 127) // 128
    codes = torch.full((nbytes + odd + 2,), 0xAA, dtype=torch.uint8, device=cuda)
    scales = torch.zeros(nblk, device=cuda)
    xd, stream = x.to(cuda), torch.cuda.current_stream().cuda_stream
    _lib.check(L.q4adamw_quantize(xd.data_ptr(), n, which, codes.data_ptr() + odd, scales.data_ptr(), stream), "quantize")
    rc, rs = oc.quant(x.numpy(), which)
    got = codes.cpu().numpy()
    assert np.array_equal(bits(scales.cpu().numpy()), bits(rs))
    assert np.array_equal(got[odd:odd + nbytes], rc)
    assert (got[:odd] == 0xAA).all() and (got[odd + nbytes:] == 0xAA).all()
    out = torch.full((n + 4,), 7.0, device=cuda)
    _lib.check(L.q4adamw_dequantize(codes.data_ptr() + odd, scales.data_ptr(), n, which, out.data_ptr(), stream), "dequantize")
    assert np.array_equal(bits(out[:n].cpu().numpy()), bits(oc.dequant(rc, rs, n, which)))
    assert bool((out[n:] == 7.0).all())


@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 1), (3000, 1), (1366, 2), (1365, 3), (77, 5), (1000, 7), (33, 256), (65, 257), (40, 1031), (300, 520)])
def test_matrices(cuda, rows, cols):
    gen = torch.Generator().manual_seed(rows * 31 + cols)
    x = grads_config1(gen, rows * cols).square().view(rows, cols)
    x[rows // 2] *= 1e-34          # scales below the reciprocal's range
    if rows > 3 and cols > 1:
        x[1] = 0.0
        x[:, cols - 1] = 0.0
        x[2, 0] = float("nan")
    codes, rmax, cmax = q.quantize_state_rank1(x.to(cuda))
    rc, rr, rcm = ot.quantize_rank1(x)
    assert torch.equal(rmax.cpu().view(torch.int32), rr.view(torch.int32))
    assert torch.equal(cmax.cpu().view(torch.int32), rcm.view(torch.int32))
    assert torch.equal(codes.cpu(), rc)
    assert torch.equal(q.quantize_state_rank1_scaled(x.to(cuda), rmax, cmax).cpu(), rc)
    # given scales smaller than the values: quotients beyond 1 get the top code
    small = q.quantize_state_rank1_scaled(x.to(cuda), rmax * 0.125, cmax * 0.125).cpu()
    quotient = x.div(ot.rank1_scale(rr * 0.125, rcm * 0.125))
    want = torch.bucketize(torch.nan_to_num(quotient, nan=-2.0, posinf=float("inf")), ot.QMID[1], right=False)
    assert torch.equal(small, ot.pack(want.reshape(-1), x.numel()))
    back = q.dequantize_state_rank1(codes, rmax, cmax)
    want = ot.dequantize_rank1(rc, rr, rcm)
    assert torch.equal(back.cpu().reshape(-1).view(torch.int32), want.reshape(-1).view(torch.int32))


@pytest.mark.parametrize("rows,cols", [(64, 40), (33, 7), (9, 1030)])
def test_statistics_that_are_no_maxima(cuda, rows, cols):
    """A caller's row and column scales are taken as numbers: the lesser of the two is the scale also
    where one of them is negative or -0.0, and a NaN beside a number gives way to it."""
    gen = torch.Generator().manual_seed(rows)
    x = grads_config1(gen, rows * cols).square().view(rows, cols)
    r, c = torch.rand(rows, generator=gen) * 1e-2 + 1e-3, torch.rand(cols, generator=gen) * 1e-2 + 1e-3
    r[3], r[5], r[7] = -0.0, -1e-3, float("nan")
    c[2], c[4], c[6] = -0.0, -2e-3, float("nan")
    scale = torch.fmin(r[:, None].expand(rows, cols), c[None, :].expand(rows, cols))
    codes = torch.randint(0, 256, ((rows * cols + 1) // 2,), dtype=torch.uint8, generator=gen)
    if rows * cols % 2:
        codes[-1] &= 15
    nibbles = torch.stack((codes & 15, codes >> 4), 1).reshape(-1)[:rows * cols].long()
    want = (ot.QMAP[1][nibbles] * scale.reshape(-1)).view(rows, cols)
    got = q.dequantize_state_rank1(codes.to(cuda), r.to(cuda), c.to(cuda)).cpu()
    number = ~torch.isnan(want)
    assert torch.equal(torch.isnan(got), ~number)
    assert torch.equal(got[number].view(torch.int32), want[number].view(torch.int32))
    want = torch.bucketize(torch.nan_to_num(x.div(scale), nan=-2.0, posinf=float("inf")), ot.QMID[1], right=False)
    got = q.quantize_state_rank1_scaled(x.to(cuda), r.to(cuda), c.to(cuda)).cpu()
    assert torch.equal(got, ot.pack(want.reshape(-1), rows * cols))
