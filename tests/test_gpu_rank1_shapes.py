"""The statistics kernels of rank-1 scaling at the sizes where their forms change or end: the
flat form up to 256 columns, or 88 where they are a multiple of 8 (a tile is 4096 / (cols | 1) rows),
the wide forms above it, and the leading statistics of tensors with several
leading dimensions, whose rows fill part of a tile, one tile or several."""
import pytest
import torch

from oracle import q4_oracle_torch as ot
from quantfour_adamw_cuda_amd import quantfour_hip as q
from tests import test_gpu_rank1 as base
from tests.q4_testlib import HP, grads_config1

pytestmark = pytest.mark.gpu

# a tile's rows: 1365 for 2 and 3 columns, 240 for 16, 31 for 128 .. 131, 16 for 255, 15 for 256
MATRICES = [(1365, 3), (1366, 2), (4100, 3), (240, 16), (241, 16), (31, 128), (63, 129), (17, 255), (46, 256),
            (300, 257), (257, 263), (64, 264), (260, 511), (9, 513), (258, 1025), (70, 1031),
            # multiples of 8 on either side of the wide form's first width, fewer rows than a tile and more
            (33, 88), (1000, 88), (33, 96), (1000, 96), (260, 104)]
# where a workgroup's rows double (6144, 24576 and 98304 rows): several tiles of the flat form, more rows of the
# wide ones; the last workgroup with all of its tiles, with some, with part of one
TALL = [(6145, 50), (6144 + 63 * 5, 64), (6200, 255), (24577, 33), (24640, 88), (98305, 24), (98304 + 500, 41), (6150, 96), (24600, 104), (98310, 96), (6200, 257)]
# the wide forms' lanes have two parts of 4 columns each under fp32 gradients, 256 columns apart: rows that end in
# either part, on its first and last columns and between them; 130 and 136 tiles, of which 128 are dealt in runs of 8
PARTS = [(37, 258), (37, 259), (40, 260), (37, 261), (40, 504), (37, 507), (40, 508), (37, 510), (40, 512), (37, 515), (40, 520), (37, 767),
         (37, 770), (2080, 520), (1088, 1541),
         # codes in windows of 4 bytes, which end the matrix' last byte and begin its first: rows that begin at either nibble
         (1, 257), (2, 257), (3, 259), (2, 261), (1, 263), (2, 511), (1, 513), (3, 1031),
         # few rows and many tiles along them: more than 256, and on either side of the rule for their statistics (3072 tiles)
         (1, 131584), (8, 131073), (9, 131073), (3, 131585), (1, 1572864), (1, 1572865), (8, 1573380), (9, 1573376)]
TENSORS = [(5, 300, 3, 3), (2, 700, 3), (1400, 1, 2), (300, 2, 7), (16, 16, 16), (3, 100, 260), (2, 130, 4, 257), (64, 3, 7, 7),
           # fewer elements below an index than a lane's; runs that end within a lane's; the most columns; half a round of
           # indices, a round and one more
           (3, 1, 2), (70, 2, 3), (700, 1, 3), (40, 1, 1, 5), (33, 90, 256), (17, 5, 2, 255), (16, 30, 3, 3), (129, 57, 3, 3), (5, 171, 3),
           # many indices with few elements below them: 64, 128 and 256 of them in a workgroup, and one more
           (49153, 1, 3), (98305, 1, 1, 7), (196609, 1, 2), (196609, 3, 3),
           # fp32 gradients, few indices: two, four and sixteen runs in a workgroup, the last of which end early; so many rows in a
           # run that the workgroup's 256 stop it at two; a third dimension with fewer and with more indices than rows; two
           # workgroups along the first dimension
           (2, 3073, 128), (1, 12517, 64), (5, 197000, 2), (1, 1025, 3, 130), (1, 11, 300, 129), (33, 800, 255)]


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16"), ("fp32", "fp16")])
@pytest.mark.parametrize("shape", MATRICES)
def test_statistics_of_a_matrix(cuda, shape, p_dt, g_dt):
    base.test_rank1_against_oracle(cuda, p_dt, g_dt, shape)


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("shape", PARTS)
def test_statistics_of_rows_that_end_anywhere_in_a_tile(cuda, shape, p_dt, g_dt):
    base.test_rank1_against_oracle(cuda, p_dt, g_dt, shape)


# the update of rows of any length: rows shorter than a lane's elements, rows that begin at each of a lane's
# elements, a matrix that ends with a row's first element in a lane, and rows of a tile and a little more or less
@pytest.mark.parametrize("stochastic", [False, True])
@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("shape", [(41, c) for c in (2, 3, 5, 6, 7, 9, 10, 11, 12, 13, 14, 15, 17, 255, 257, 261, 511, 513, 514, 515)])
def test_update_of_rows_that_begin_anywhere_in_a_lane(cuda, shape, p_dt, g_dt, stochastic):
    test = base.test_rank1_stochastic_rounding_against_oracle if stochastic else base.test_rank1_against_oracle
    test(cuda, p_dt, g_dt, shape)


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("shape", TALL)
def test_statistics_of_a_tall_matrix(cuda, shape, p_dt, g_dt):
    base.test_rank1_against_oracle(cuda, p_dt, g_dt, shape)


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("shape", TENSORS)
def test_statistics_of_several_dimensions(cuda, shape, p_dt, g_dt):
    base.test_rank1_more_than_two_dimensions_against_oracle(cuda, shape, p_dt, g_dt, False)


def test_statistics_of_many_indices_of_the_first_dimension(cuda):
    """Enough elements that a workgroup takes 64 indices (12.6 million), the last one 8 of them; the oracle on the GPU."""
    shape = (200, 7000, 3, 3)
    gen = torch.Generator(device=cuda).manual_seed(5)
    n, rows = 12_600_000, 4_200_000
    z = lambda m, dt=torch.float32: torch.zeros(m, dtype=dt, device=cuda)
    p0 = torch.randn(shape, generator=gen, device=cuda) * 0.05
    p, m, v, sm = p0.clone(), z(n // 2, torch.uint8), z(n // 2, torch.uint8), z((n + 127) // 128)
    r, rn, c, cn = z(rows), z(rows), z(3), z(3)
    lead = ([z(d) for d in shape[:-1]], [z(d) for d in shape[:-1]])
    ref = (p0, m.clone(), v.clone(), sm.clone(), [z(200).view(200, 1, 1, 1), z(7000).view(1, 7000, 1, 1), z(3).view(1, 1, 3, 1), z(3).view(1, 1, 1, 3)])
    for step in (1, 2):
        g = torch.randn(shape, generator=gen, device=cuda) * torch.rand(200, 1, 1, 1, generator=gen, device=cuda)
        with torch.no_grad():
            ref = ot.step_quant_rank1_nd(ref[0], g, *ref[1:], step=step, **HP)
        q.fused_4bit_rank1_multi([p], [g], [m], [v], [sm], [r], [c], [rn], [cn], *base.HPA, step, leads=[lead])
        for have, want in zip(lead[0] + [c], ref[4]):
            assert torch.equal(have, want.reshape(-1)), f"step {step}: statistics"
        assert torch.equal(m, ref[1]) and torch.equal(v, ref[2]), f"step {step}: codes"


@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "bf16"), ("bf16", "bf16")])
@pytest.mark.parametrize("copies", [1, 9])
def test_one_list_of_every_form(cuda, copies, p_dt, g_dt):
    """Matrices and tensors of every statistics kernel side by side in one call, several kinds to a batch, in
    one batch of an update kernel and in more: each equals the oracle's, and the steps are the same as one by one."""
    shapes = [(40, 64), (3, 5, 64), (36, 400), (33, 77), (30, 301), (4, 6, 7), (66, 1024), (20, 520), (2, 9, 264), (5, 3, 3, 3)] * copies
    gen = torch.Generator().manual_seed(copies)
    z = lambda n, dt=torch.float32: torch.zeros(n, dtype=dt, device=cuda)

    def state(p):
        n, cols = p.numel(), p.shape[-1]
        lead = [z(d) for d in p.shape[:-1]] if p.dim() > 2 else None
        return dict(p=p.clone().to(cuda), m=z((n + 1) // 2, torch.uint8), v=z((n + 1) // 2, torch.uint8), sm=z((n + 127) // 128),
                    r=z(n // cols), c=z(cols), rn=z(n // cols), cn=z(cols), lead=lead and (lead, [torch.zeros_like(x) for x in lead]))

    def call(ss, gs, step):
        pick = lambda k: [s[k] for s in ss]
        q.fused_4bit_rank1_multi(pick("p"), [g.clone() for g in gs], pick("m"), pick("v"), pick("sm"), pick("r"), pick("c"), pick("rn"),
                                 pick("cn"), *base.HPA, step, leads=pick("lead"))

    ps = [(torch.randn(s, generator=gen) * 0.05).to(base.DT[p_dt]) for s in shapes]
    together, alone = [state(p) for p in ps], [state(p) for p in ps]
    refs = [(p, z((p.numel() + 1) // 2, torch.uint8).cpu(), z((p.numel() + 1) // 2, torch.uint8).cpu(), z((p.numel() + 127) // 128).cpu(),
             [torch.zeros([p.shape[j] if d == j else 1 for d in range(p.dim())]) for j in range(p.dim())]) for p in ps]
    for step in (1, 2):
        gs = [grads_config1(gen, p.numel()).view(p.shape).to(base.DT[g_dt]) for p in ps]
        dev = [g.to(cuda) for g in gs]
        call(together, dev, step)
        for i, s in enumerate(alone):
            call([s], [dev[i]], step)
            refs[i] = ot.step_quant_rank1_nd(refs[i][0], gs[i], *refs[i][1:], step=step, **HP)
            t = together[i]
            for k in ("p", "m", "v", "sm", "r", "c"):
                assert torch.equal(s[k].view(torch.uint8), t[k].view(torch.uint8)), f"{shapes[i]} step {step}: {k} alone and together"
            assert torch.equal(t["m"].cpu(), refs[i][1]) and torch.equal(t["v"].cpu(), refs[i][2]), f"{shapes[i]} step {step}: codes"
            stats = (t["lead"][0] if t["lead"] else [t["r"]]) + [t["c"]]
            for have, want in zip(stats, refs[i][4]):
                assert torch.equal(have.cpu().view(torch.int32), want.reshape(-1).view(torch.int32)), f"{shapes[i]} step {step}: statistics"
            assert not t["rn"].any() and not t["cn"].any()


@pytest.mark.parametrize("stochastic", [False, True])
@pytest.mark.parametrize("p_dt,g_dt", [("fp32", "fp32"), ("bf16", "bf16")])
@pytest.mark.parametrize("shape", [(7, 1, 2), (1, 9, 2), (40, 60, 2), (2, 3, 400, 2), (3, 1, 50, 3), (6, 70, 1, 5), (9, 40, 3, 3), (2, 5, 7, 63),
                                   (33, 31, 61), (5, 130, 8), (4, 11, 65)])
def test_short_rows_of_several_dimensions(cuda, shape, p_dt, g_dt, stochastic):
    """The kernel that makes the rows' scales from the leading statistics: rows of two elements (more of them than a
    workgroup's threads take at once), leading dimensions of one index, the longest rows and the first
    beyond them; gradients whose second moments lie below and above the reciprocals' range, which
    sends elements to the division.  The rows' scales that the step leaves are the statistics' minima."""
    gen = torch.Generator().manual_seed(sum(shape) + stochastic)
    n, cols, k = int(torch.Size(shape).numel()), shape[-1], len(shape) - 1
    rows = n // cols
    z = lambda m, dt=torch.float32: torch.zeros(m, dtype=dt, device=cuda)
    p0 = (torch.randn(shape, generator=gen) * 0.05).to(base.DT[p_dt])
    p, m, v, sm = p0.clone().to(cuda), z((n + 1) // 2, torch.uint8), z((n + 1) // 2, torch.uint8), z((n + 127) // 128)
    r, rn, c, cn = z(rows), z(rows), z(cols), z(cols)
    lead = ([z(d) for d in shape[:-1]], [z(d) for d in shape[:-1]])
    ref = (p0, m.cpu(), v.cpu(), sm.cpu(), [torch.zeros([shape[j] if d == j else 1 for d in range(k + 1)]) for j in range(k + 1)])
    sr = dict(seed=0x1234_5678_9ABC, tensor_salt=3) if stochastic else {}
    for step, scale in ((1, 1.0), (2, 1e-17), (3, 1e17), (4, 1.0)):
        g = grads_config1(gen, n).view(shape) * 1e3
        g[shape[0] // 2:] *= scale                  # half of the first dimension: scales of both kinds meet
        g = g.to(base.DT[g_dt])
        if step == 2:                               # the second moments are small only where no large ones are left
            ref = (ref[0], ref[1], torch.zeros_like(ref[2]), ref[3], [torch.zeros_like(x) for x in ref[4]])
            for x in (v, r, c, *lead[0]):
                x.zero_()
        with torch.no_grad():
            ref = ot.step_quant_rank1_nd(ref[0], g, *ref[1:], step=step, **sr, **HP)
        q.fused_4bit_rank1_multi([p], [g.to(cuda)], [m], [v], [sm], [r], [c], [rn], [cn], *base.HPA, step, leads=[lead],
                                 **(dict(seed=sr["seed"], salts=[3]) if stochastic else {}))
        what = f"{shape} {p_dt}/{g_dt} step {step}"
        assert torch.equal(m.cpu(), ref[1]), f"{what}: m codes"
        for have, want in zip(lead[0] + [c], ref[4]):
            assert torch.equal(have.cpu().view(torch.int32), want.reshape(-1).view(torch.int32)), f"{what}: statistics"
        assert torch.equal(v.cpu(), ref[2]), f"{what}: v codes"
        assert torch.equal(r, q.rank1_row_scale(lead[0], shape[:-1])), f"{what}: rows' scales"
        assert not rn.any() and not cn.any() and not any(x.any() for x in lead[1]), f"{what}: scratch"


@pytest.mark.parametrize("stochastic", [False, True])
@pytest.mark.parametrize("g_dt", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("shape", [(300, 3), (77, 50), (1000, 88), (6200, 41), (64, 264), (33, 301),
                                   (5, 40, 3, 3), (33, 7, 5), (20, 3, 64), (3, 9, 264), (2, 5, 300), (2, 3, 300, 3), (3, 2, 270, 40),
                                   (2, 3073, 128)])
def test_multiplier_and_non_finite_gradients(cuda, shape, g_dt, stochastic):
    """Every statistics kernel with a device multiplier (gradients scaled up by it, so that the product is
    exact) and cleared gradients; NaN and infinities in the second step: maxima are taken over the
    non-NaN values, a finite value under an infinite scale and a NaN get code 0."""
    gen = torch.Generator().manual_seed(sum(shape))
    n, cols, k = int(torch.Size(shape).numel()), shape[-1], len(shape) - 1
    rows = n // cols
    z = lambda m, dt=torch.float32: torch.zeros(m, dtype=dt, device=cuda)
    p0 = torch.randn(shape, generator=gen) * 0.05
    p, m, v, sm = p0.clone().to(cuda), z((n + 1) // 2, torch.uint8), z((n + 1) // 2, torch.uint8), z((n + 127) // 128)
    r, rn, c, cn = z(rows), z(rows), z(cols), z(cols)
    lead = ([z(d) for d in shape[:-1]], [z(d) for d in shape[:-1]]) if k > 1 else None
    ref = (p0, m.cpu(), v.cpu(), sm.cpu(), [torch.zeros([shape[j] if d == j else 1 for d in range(k + 1)]) for j in range(k + 1)])
    scale = torch.tensor([0.0625], device=cuda)
    sr = dict(seed=0xABCD_1234_5678, tensor_salt=2) if stochastic else {}
    for step in (1, 2, 3):
        g = grads_config1(gen, n).view(shape)
        if step == 2:
            flat = g.view(-1)
            flat[n // 3], flat[n // 2], flat[n // 2 + 1], flat[n - 1] = float("inf"), float("nan"), float("-inf"), float("nan")
            g.view(rows, cols)[rows // 4] = float("nan")
        g = g.to(base.DT[g_dt]) * 16          # a power of two: the multiplier takes it back exactly
        with torch.no_grad():
            ref = ot.step_quant_rank1_nd(ref[0], g.float() * 0.0625, *ref[1:], step=step, **sr, **HP)
        dg = g.to(cuda)
        q.fused_4bit_rank1_multi([p], [dg], [m], [v], [sm], [r], [c], [rn], [cn], *base.HPA, step, grad_scale_dev=scale, zero_grad=True,
                                 leads=[lead], **(dict(seed=sr["seed"], salts=[2]) if stochastic else {}))
        what = f"{shape} {g_dt} step {step}"
        assert not dg.any(), f"{what}: gradients not cleared"
        assert torch.equal(m.cpu(), ref[1]), f"{what}: m codes"
        assert torch.equal(sm.cpu().view(torch.int32), ref[3].view(torch.int32)), f"{what}: m scales"
        for have, want in zip((lead[0] if lead else [r]) + [c], ref[4]):
            assert torch.equal(have.cpu().view(torch.int32), want.reshape(-1).view(torch.int32)), f"{what}: statistics"
        assert torch.equal(v.cpu(), ref[2]), f"{what}: v codes"
        assert not rn.any() and not cn.any(), f"{what}: scratch"
