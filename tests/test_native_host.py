"""The native host code (csrc/q4host.cpp): it takes the common case and leaves everything else to the Python
code, with the same results."""
import ctypes

import pytest
import torch

from quantfour_adamw_cuda_amd import AdamWFused_QuantFour, _lib
from quantfour_adamw_cuda_amd import quantfour_hip as q

HP = (0.9, 0.999, 1e-3, 0.01, 1e-8)


def test_what_is_not_for_it_is_left_alone():
    _lib.load()
    h = _lib.host
    p, g = torch.zeros(200), torch.zeros(200)
    state = [torch.zeros(100, dtype=torch.uint8), torch.zeros(100, dtype=torch.uint8), torch.zeros(2), torch.zeros(2)]
    assert h.fused_4bit(p, g, *state, *HP, 1.0) is None                    # not on a GPU
    assert h.fused_4bit(p, None, *state, *HP, 1.0) is None and h.fused_4bit(p, g) is None
    assert h.fused_single_tensor(p, g, p, g, *HP, 1.0) is None
    par = torch.nn.Parameter(torch.zeros(4))
    par.grad = torch.zeros(4)
    table = (_lib.Q4Grad * 2)()
    assert h.gradients(([par],), ctypes.addressof(table), 2) is None and h.gradients(([],), ctypes.addressof(table), 2) is None
    assert h.plan((par,), torch.zeros(1), [], [], []) is None
    with pytest.raises((TypeError, ValueError)):
        h.refresh(object(), [par], torch.zeros(1))
    with pytest.raises(TypeError):
        h.run(1)


def _twins(cuda, shapes, p_dt, g_dt, **kw):
    gen = torch.Generator(device=cuda).manual_seed(3)
    sides = []
    base = [(torch.randn(s, generator=gen, device=cuda) * 0.05).to(p_dt) for s in shapes]
    for native in (True, False):
        ps = [torch.nn.Parameter(b.clone()) for b in base]
        for p in ps:
            if p_dt != g_dt:
                p.grad_dtype = g_dt
        opt = AdamWFused_QuantFour(ps, lr=1e-3, weight_decay=0.01, **kw)
        if not native:
            opt._make_native = lambda plan: None
            opt._one_norm = lambda *a: None
        sides.append((ps, opt))
    return gen, sides


@pytest.mark.gpu
@pytest.mark.parametrize("p_dt,g_dt", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16)])
@pytest.mark.parametrize("kw", [{}, dict(round_type="stochastic", seed=5), dict(variance_scale_type="rank1"),
                                dict(variance_scale_type="rank1", round_type="stochastic", seed=2 ** 40 + 1)])
def test_steps_equal_the_python_codes(cuda, kw, p_dt, g_dt):
    """Every kind of launch, new gradient tensors each step, options of a step, a learning rate that changes, a
    parameter without a gradient in one step."""
    gen, sides = _twins(cuda, [(70, 129), (5000,), (64, 512), (100,), (3, 20, 96), (30, 16, 3, 3)], p_dt, g_dt, **kw)
    options = [{}, dict(max_grad_norm=0.5), dict(grad_scale=0.25, zero_grad=True), dict(found_inf=torch.ones(1, device=cuda)),
               dict(grad_scale=torch.full((1,), 2.0, device=cuda), max_grad_norm=3.0, found_inf=torch.zeros(1, device=cuda)), {}, {}]
    for step, more in enumerate(options):
        gs = [(torch.randn(p.shape, generator=gen, device=cuda) * 1e-2).to(g_dt) for p in sides[0][0]]
        for ps, opt in sides:
            opt.param_groups[0]["lr"] = 1e-3 * (1 + step)
            for i, (p, g) in enumerate(zip(ps, gs)):
                p.grad = None if step == 5 and i == 2 else g.clone()
            opt.step(**more)
        assert sides[0][1]._plans[0].native is not None and sides[1][1]._plans[0].native is None
        for (pa, pb) in zip(sides[0][0], sides[1][0]):
            assert torch.equal(pa.view(torch.uint8), pb.view(torch.uint8)), f"step {step}: {tuple(pa.shape)}"
            assert pb.grad is None or torch.equal(pa.grad, pb.grad)
        if "max_grad_norm" in more:
            assert torch.equal(sides[0][1].last_grad_norm, sides[1][1].last_grad_norm)
    a, b = (opt.state_dict()["state"] for _, opt in sides)
    for i in a:
        assert float(a[i]["step"]) == float(b[i]["step"]) == (5.0 if i == 2 else 6.0)
        assert torch.equal(a[i]["exp_avg"], b[i]["exp_avg"]) and torch.equal(a[i]["exp_avg_sq"], b[i]["exp_avg_sq"])


@pytest.mark.gpu
@pytest.mark.parametrize("small,kinds", [(59, ["fused_4bit"]), (60, ["fused_4bit", "fused_single_tensor"])])
@pytest.mark.parametrize("kw", [{}, dict(round_type="stochastic", seed=5)])
def test_timed_steps_make_the_same_launches(cuda, kw, small, kinds):
    """Steps with launch timing, which the Python code makes, against steps without: one launch for both kinds up to 61
    tensors, and for tensors of one step number only; the same results."""
    gen, ((pa, timed), (pb, plain)) = _twins(cuda, [(70, 129), (5000,)] + [(100 + i,) for i in range(small)], torch.float32, torch.float32, **kw)
    plain._make_native, plain._one_norm = type(plain)._make_native.__get__(plain), type(plain)._one_norm.__get__(plain)
    for step in range(4):
        gs = [torch.randn(p.shape, generator=gen, device=cuda) * 1e-2 for p in pa]
        timed.kernel_timing = []
        for ps, opt in ((pa, timed), (pb, plain)):
            for i, (p, g) in enumerate(zip(ps, gs)):
                p.grad = None if step == 1 and i < 2 else g      # the quantized ones lag by a step from here on
            opt.step(zero_grad=False)
        seen = sorted(kind for kind, _, _ in timed.kernel_timing)
        assert seen == (kinds if step == 0 else ["fused_single_tensor"] if step == 1 else ["fused_4bit", "fused_single_tensor"]), f"step {step}"
        assert plain._plans[0].native is not None
        for a, b in zip(pa, pb):
            assert torch.equal(a, b), f"step {step}: {tuple(a.shape)}"
            for key in ("exp_avg", "exp_avg_sq"):
                assert torch.equal(timed.state[a][key], plain.state[b][key])


@pytest.mark.gpu
def test_refusals_are_the_python_codes(cuda):
    n = 5000
    nbytes, nblk = q.state_sizes(n)
    z = lambda k, dt=torch.float32: torch.zeros(k, dtype=dt, device=cuda)
    p, g, m, v, sm, sv = z(n), z(n), z(nbytes, torch.uint8), z(nbytes, torch.uint8), z(nblk), z(nblk)
    for bad, words in (((p, g[:-1], m, v, sm, sv), "grad numel"), ((p, z(2 * n)[::2], m, v, sm, sv), "grad must be contiguous"),
                       ((p, g, m[:-1], v, sm, sv), "packed size"), ((p, g, m, v, sm, sv.double()), "scales must be float32"),
                       ((p, g.cpu(), m, v, sm, sv), "grad must be on")):
        with pytest.raises(AssertionError, match=words):
            q.fused_4bit(*bad, *HP, 1)
    with pytest.raises(TypeError, match="float32, bfloat16 or float16"):
        q.fused_4bit(p.double(), g, m, v, sm, sv, *HP, 1)
    with pytest.raises(RuntimeError, match="hyper-parameter"):
        q.fused_4bit(p, g, m, v, sm, sv, 1.5, 0.999, 1e-3, 0.01, 1e-8, 1)
    q.fused_4bit(p, g, m, v, sm, sv, *HP, torch.tensor(1.0))      # anything float() takes
    opt = AdamWFused_QuantFour([torch.nn.Parameter(z(n))], lr=1e-3)
    par = opt.param_groups[0]["params"][0]
    par.grad = z(n)
    opt.step()
    opt.param_groups[0]["eps"] = -1.0
    with pytest.raises(RuntimeError, match="fused_4bit_multi failed"):
        opt.step()
    opt.param_groups[0]["eps"] = 1e-8
    par.grad = z(2 * n)[:n]
    par.grad.as_strided_((n,), (2,))                              # re-strided in place: no longer dense
    with pytest.raises(AssertionError, match="grad must be contiguous"):
        opt.step()


@pytest.mark.gpu
@pytest.mark.parametrize("p_dt,g_dt", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("stochastic", [False, True])
@pytest.mark.parametrize("quantized,small", [(1, 1), (5, 56), (5, 57), (0, 3), (3, 0)])
def test_one_call_for_both_kinds(cuda, quantized, small, stochastic, p_dt, g_dt):
    """q4adamw_fused_step_multi against the calls it stands for, bit for bit: 61 tensors, which are one launch, and 62;
    small tensors of a part of a workgroup, of one, of more; a multiplier, cleared gradients, a cancelled step."""
    L = _lib.load()
    gen = torch.Generator(device=cuda).manual_seed(quantized * 100 + small)
    q_sizes = [(5000, 128, 4097, 2048, 70001)[i % 5] + i for i in range(quantized)]
    s_sizes = [(1, 255, 256, 1024, 1025, 2047, 2049, 4096, 9000)[i % 9] for i in range(small)]
    tag = q._DTYPE_TAG
    stream = q._stream(torch.device("cuda", torch.cuda.current_device()))
    salts = q.make_salts([7 * i + 1 for i in range(quantized)]) if quantized else None
    scale, skip = torch.full((1,), 0.5, device=cuda), torch.ones(1, device=cuda)
    base = [(torch.randn(n, generator=gen, device=cuda) * 0.05).to(p_dt) for n in q_sizes + s_sizes]

    def side():
        ps = [b.clone() for b in base]
        z = lambda n, dt=torch.float32: torch.zeros(n, dtype=dt, device=cuda)
        qs = [(z(nb, torch.uint8), z(nb, torch.uint8), z(nk), z(nk)) for nb, nk in map(q.state_sizes, q_sizes)]
        return ps, qs, [(z(n), z(n)) for n in s_sizes]

    one, two = side(), side()
    for step, opts in ((1, {}), (2, dict(grad_scale_dev=scale, zero_grad=True)), (3, dict(found_inf=skip, zero_grad=True)), (4, {})):
        gs = [(torch.randn(n, generator=gen, device=cuda) * 1e-2).to(g_dt) for n in q_sizes + s_sizes]
        kept = []
        for k, (ps, qs, ss) in enumerate((one, two)):
            g = [x.clone() for x in gs]
            kept.append(g)
            qt = q.make_table(ps[:quantized], g[:quantized], *([x[j] for x in qs] for j in range(4)))
            st = q.make_small_table(ps[quantized:], g[quantized:], [x[0] for x in ss], [x[1] for x in ss])
            o = q.grad_options(scale.device, **opts)
            tail = (tag[p_dt], tag[g_dt], *HP[:5], float(step), o, stream)
            if k == 0:
                _lib.check(L.q4adamw_fused_step_multi(qt, quantized, st, small, int(stochastic), salts, 99, *tail), "fused_step_multi")
            else:
                _lib.check(L.q4adamw_fused_single_tensor_multi_ex(st, small, *tail), "small")
                if stochastic:
                    _lib.check(L.q4adamw_fused_4bit_multi_sr(qt, quantized, salts, 99, *tail), "sr")
                else:
                    _lib.check(L.q4adamw_fused_4bit_multi_ex(qt, quantized, *tail), "ex")
        for a, b in zip(kept[0] + one[0] + [t for s in one[1] + one[2] for t in s], kept[1] + two[0] + [t for s in two[1] + two[2] for t in s]):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), f"step {step}"


@pytest.mark.gpu
@pytest.mark.parametrize("small", [2, 3])
def test_one_call_at_the_most_workgroups(cuda, small):
    """One launch takes both kinds up to 2^17 workgroups of 1024 elements; a list of one more takes two."""
    L = _lib.load()
    gen = torch.Generator(device=cuda).manual_seed(small)
    n = ((1 << 17) - 2) * 1024 - 100                     # 2^17 - 2 workgroups, one more for every small tensor
    z = lambda k, dt=torch.float32: torch.zeros(k, dtype=dt, device=cuda)
    nb, nk = q.state_sizes(n)
    stream = q._stream(torch.device("cuda", torch.cuda.current_device()))
    base = [torch.randn(k, generator=gen, device=cuda) * 0.05 for k in [n] + [700] * small]
    gs = [(torch.randn(b.numel(), generator=gen, device=cuda) * 1e-2).to(torch.bfloat16) for b in base]
    sides = []
    for one in (True, False):
        ps = [b.clone() for b in base]
        qs, ss = [z(nb, torch.uint8), z(nb, torch.uint8), z(nk), z(nk)], [(z(700), z(700)) for _ in range(small)]
        qt = q.make_table(ps[:1], gs[:1], *([x] for x in qs))
        st = q.make_small_table(ps[1:], gs[1:], [x[0] for x in ss], [x[1] for x in ss])
        tail = (0, 1, *HP, 1.0, None, stream)
        if one:
            _lib.check(L.q4adamw_fused_step_multi(qt, 1, st, small, 0, None, 0, *tail), "fused_step_multi")
        else:
            _lib.check(L.q4adamw_fused_single_tensor_multi_ex(st, small, *tail), "small")
            _lib.check(L.q4adamw_fused_4bit_multi_ex(qt, 1, *tail), "ex")
        sides.append(ps + qs + [t for s in ss for t in s])
    for a, b in zip(*sides):
        assert torch.equal(a, b)
    assert all(not torch.equal(p, b) for p, b in zip(sides[0], base))


class _Named(torch.Tensor):
    """A tensor subclass, as programs make them to carry a name along."""


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["parameter", "gradient"])
def test_tensor_subclasses(cuda, where):
    """A parameter of a subclass keeps its group on the Python path, a gradient of one is the memory that it is: the same
    results as plain tensors."""
    gen, ((pa, a), (pb, b)) = _twins(cuda, [(70, 129), (100,)], torch.float32, torch.float32)
    if where == "parameter":
        pa[0] = torch.nn.Parameter(pa[0].detach().as_subclass(_Named))
        a = AdamWFused_QuantFour(pa, lr=1e-3, weight_decay=0.01)
        assert isinstance(pa[0], _Named)
    for step in range(3):
        for x, y in zip(pa, pb):
            g = torch.randn(y.shape, generator=gen, device=cuda) * 1e-2
            x.grad = g.clone().as_subclass(_Named) if where == "gradient" else g.clone()
            y.grad = g
        a.step(max_grad_norm=0.5)
        b.step(max_grad_norm=0.5)
        if where == "parameter":
            assert a._plans[0].native is None
        for x, y in zip(pa, pb):
            assert torch.equal(x.detach().as_subclass(torch.Tensor), y.detach()), f"step {step}"
