"""The optimizer's workloads, for timing and for comparing results: what a training program has
it do, from one small tensor to parameter sets of billions of elements.

Three kinds of work:

  step    one `AdamWFused_QuantFour.step()` over a parameter set in the middle of training (its
          state has seen two steps), with gradients in place
  call    one `fused_4bit` / `fused_single_tensor` call on one tensor, for programs that keep
          their own state and do without the optimizer class
  encode, decode
          both moments of one tensor from fp32 to the packed form and back: what
          taking over a torch.optim.AdamW checkpoint, and handing one out, does per tensor

A parameter set's tensors, and each kind of their state, lie one after another in a flat buffer
(every tensor on a 256-byte boundary, as the caching allocator places them), so that parameters,
codes, scales and statistics come back whole in a few outputs.
"""
import math
import random

import torch

from quantfour_adamw_cuda_amd import (AdamWFused_QuantFour, dequantize_state, fused_4bit, fused_single_tensor,
                                      quantize_state, state_sizes)
from quantfour_adamw_cuda_amd import quantfour_hip

HP = dict(lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.01)
THRESHOLD = 4096          # tensors of at most this many elements keep fp32 moments
LARGEST = 2_000_000_000   # elements: no case has more
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
SIZE = {"float32": 4, "bfloat16": 2, "float16": 2}


# -- parameter sets -----------------------------------------------------------
def shapes_of(case):
    """The shapes of a step case's parameter set."""
    kind, layers = case["set"], case.get("layers", 0)
    if kind == "mlp":             # linear layers with biases, `width` wide
        w = case["width"]
        return [(w, 4), (w,)] + [s for _ in range(layers) for s in ((w, w), (w,))] + [(1, w), (1,)]
    if kind == "matrix":
        return [(case["rows"], case["cols"])]
    if kind == "ragged":          # lengths around the block size and the quantization threshold, two long ones
        r = random.Random(case["pick"])
        odd = case["longest"] | 1
        return ([(1,), (127,), (128,), (129,), (4095,), (4097,)]
                + [(r.randint(1, 20000),) for _ in range(case["more"])] + [(odd,), (3, odd)])
    if kind == "gpt2-small":
        s = [(50257, 768), (1024, 768)]
        for _ in range(layers):
            s += [(768,), (768,), (768, 2304), (2304,), (768, 768), (768,),
                  (768,), (768,), (768, 3072), (3072,), (3072, 768), (768,)]
        return s + [(768,), (768,)]
    if kind == "llama3-8b":       # embedding and head, then transformer layers
        s = [(128256, 4096)] * case["tables"]
        for _ in range(layers):
            s += [(4096, 4096), (1024, 4096), (1024, 4096), (4096, 4096),
                  (14336, 4096), (14336, 4096), (4096, 14336), (4096,), (4096,)]
        return s + [(4096,)]
    if kind == "llama2-13b":
        s = [(32000, 5120)] * case["tables"]
        for _ in range(layers):
            s += [(5120, 5120)] * 4 + [(13824, 5120)] * 2 + [(5120, 13824), (5120,), (5120,)]
        return s
    if kind == "convnet":         # residual blocks of 3x3 convolutions with their norms, a 7x7 stem, a classifier
        w = case["width"]
        s = [(w, 3, 7, 7), (w,), (w,)]
        c = w
        for stage in range(4):
            o = w << stage
            for b in range(layers):
                s += [(o, c, 3, 3), (o,), (o,), (o, o, 3, 3), (o,), (o,)]
                if c != o:
                    s += [(o, c, 1, 1), (o,), (o,)]
                c = o
        return s + [(1000, c), (1000,)]
    raise ValueError(kind)


def _step(name, kind, p, g, scale="group", rounding="real-nearest", clip=False, amp=False, **more):
    c = {"do": "step", "set": kind, "p": p, "g": g, "scale": scale, "round": rounding, "clip": clip, "amp": amp, **more}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest: one tensor just above the quantization threshold, called directly
        # (a program with its own state; latency of one launch)
        {"name": "call small fp32", "do": "call", "numel": 64 * 130, "p": "float32", "g": "float32"},
        # optimizer.step() of a tiny model whose tensors all keep fp32 moments: host latency
        _step("mlp tiny", "mlp", "float32", "float32", width=8, layers=1),
        # one fp32 matrix: a step of tens of microseconds, where one launch's start and end count
        _step("matrix 4096 fp32", "matrix", "float32", "float32", rows=4096, cols=4096),
        # odd lengths: tail blocks, tensors on either side of the threshold, rows of odd length
        _step("ragged fp32", "ragged", "float32", "float32", pick=0, more=0, longest=1000003),
        # a small language model trained in fp32 with global-norm clipping, as it usually is:
        # 148 tensors, half of them tiny
        _step("gpt2-small fp32 clip", "gpt2-small", "float32", "float32", clip=True, layers=12),
        # large-model training with fp32 master parameters and bf16 gradients: the main workload
        _step("llama3-8b fp32/bf16", "llama3-8b", "float32", "bfloat16", layers=4, tables=2),
        # the same with bf16 parameters: the smallest memory footprint
        _step("llama2-13b bf16", "llama2-13b", "bfloat16", "bfloat16", layers=4, tables=2),
        # bf16 parameters with stochastic rounding of the moments
        _step("llama2-13b bf16 sr", "llama2-13b", "bfloat16", "bfloat16", rounding="stochastic", layers=4, tables=2),
        # rank-1 scaling of the second moment (the 4-bit paper's default for matrices)
        _step("llama3-8b rank1", "llama3-8b", "float32", "bfloat16", scale="rank1", layers=4, tables=2),
        # rank-1 scaling of an image model: four-dimensional tensors with rows of three elements
        _step("convnet rank1", "convnet", "float32", "float32", scale="rank1", width=64, layers=2),
        # taking over an AdamW checkpoint: both moments of one large matrix
        {"name": "encode", "do": "encode", "scale": "group", "rows": 14336, "cols": 4096},
        # handing one out
        {"name": "decode", "do": "decode", "scale": "group", "rows": 14336, "cols": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    what = rng.choice(["step"] * 7 + ["call", "encode", "decode"])
    p, g = rng.choice([("float32", "float32"), ("float32", "bfloat16"), ("bfloat16", "bfloat16"), ("float32", "float16"),
                       ("float16", "float16"), ("bfloat16", "float32")])
    if what == "call":
        return {"do": "call", "numel": _log_int(rng, 64, 1 << 25), "p": p, "g": g}
    if what in ("encode", "decode"):
        cols = _log_int(rng, 32, 16384)
        if rng.random() < 0.5:
            cols = max(32, cols // 64 * 64)
        rows = max(1, _log_int(rng, 1 << 14, 1 << 27) // cols)
        return {"do": what, "scale": rng.choice(["group", "group", "rank1"]), "rows": rows, "cols": cols}
    scale = rng.choice(["group", "group", "rank1"])
    opts = dict(scale=scale, rounding=rng.choice(["real-nearest", "real-nearest", "stochastic"]),
                clip=rng.random() < 0.4, amp=rng.random() < 0.25)
    kind = rng.choice(["mlp", "matrix", "matrix", "ragged", "gpt2-small", "llama3-8b", "llama2-13b", "convnet"])
    if kind == "mlp":
        return _step("", kind, p, g, width=_log_int(rng, 4, 2048), layers=rng.randint(0, 8), **opts)
    if kind == "matrix":
        cols = _log_int(rng, 48, 16384)
        if rng.random() < 0.5:
            cols = max(64, cols // 64 * 64)
        return _step("", kind, p, g, rows=max(2, _log_int(rng, 5000, 1 << 28) // cols), cols=cols, **opts)
    if kind == "ragged":
        return _step("", kind, p, g, pick=rng.randint(1, 10 ** 6), more=rng.randint(0, 60), longest=_log_int(rng, 5001, 10 ** 7), **opts)
    if kind == "convnet":
        return _step("", kind, p, g, width=rng.choice([24, 32, 48, 64, 96]), layers=rng.randint(1, 3), **opts)
    if kind == "gpt2-small":
        return _step("", kind, p, g, layers=rng.randint(1, 12), **opts)
    return _step("", kind, p, g, layers=rng.randint(1, 4), tables=rng.randint(0, 2), **opts)


# -- inputs -------------------------------------------------------------------
def _numel(shape):
    n = 1
    for s in shape:
        n *= s
    return n


class _Flat:
    """Views of one buffer, each on a 256-byte boundary."""

    def __init__(self, sizes, dtype, device):
        step = 256 // torch.empty(0, dtype=dtype).element_size()
        at, offsets = 0, []
        for n in sizes:
            offsets.append(at)
            at += -(-n // step) * step
        self.all = torch.zeros(at, dtype=dtype, device=device)
        self.views = [self.all[o:o + n] for o, n in zip(offsets, sizes)]


def _normal(out, gen, std):
    for part in out.split(1 << 28):
        part.copy_(torch.randn(part.numel(), generator=gen, device=part.device).mul_(std))


def _gradient(out, gen, kind):
    """"heavy": Student-t with three degrees of freedom times 1e-4, as large models' gradients
    look; "outliers": N(0, 1e-3^2) with 0.1 % of +-0.1; "edges": the same normals with 20 % exact
    zeros, 1 % denormals and 0.01 % of +-1e3."""
    for part in out.split(1 << 28):
        n, dev = part.numel(), part.device
        g = torch.randn(n, generator=gen, device=dev)
        if kind == "heavy":
            c = torch.randn(n, generator=gen, device=dev).square_()
            for _ in range(2):
                c += torch.randn(n, generator=gen, device=dev).square_()
            g.mul_(c.mul_(1.0 / 3.0).rsqrt_()).mul_(1e-4)
        else:
            u = torch.rand(n, generator=gen, device=dev)
            g.mul_(1e-3)
            if kind == "outliers":
                g[u < 5e-4] = 0.1
                g[u > 1.0 - 5e-4] = -0.1
            else:
                g = torch.where(u < 0.2, 0.0, torch.where(u < 0.21, g * 1e-36, torch.where(u < 0.2101, torch.sign(g) * 1e3, g)))
        part.copy_(g)


def _prepare_step(case, gen, device):
    shapes = shapes_of(case)
    sizes = [_numel(s) for s in shapes]
    assert sum(sizes) <= LARGEST, case
    p_flat = _Flat(sizes, DTYPES[case["p"]], device)
    g_flat = _Flat(sizes, DTYPES[case["g"]], device)
    kind = {"l": "heavy", "r": "edges"}.get(case["set"][0], "outliers")
    _normal(p_flat.all, gen, 0.02)
    # tokens that training has not met yet: half of an embedding's rows never had a gradient
    unseen = None
    if case.get("tables"):
        unseen = torch.rand(shapes[0][0], generator=gen, device=device) < 0.5
    params = []
    for shape, p, g in zip(shapes, p_flat.views, g_flat.views):
        p = torch.nn.Parameter(p.view(shape))
        if case["g"] != case["p"]:
            p.grad_dtype = DTYPES[case["g"]]
        p.grad = g.view(shape)
        params.append(p)
    seed = int(torch.randint(1 << 31, (1,), generator=gen, device=device)) if case["round"] == "stochastic" else None
    opt = AdamWFused_QuantFour(params, variance_scale_type=case["scale"], round_type=case["round"], seed=seed, **HP)
    kw = {}
    if case["clip"]:
        kw["max_grad_norm"] = 1.0
    if case["amp"]:    # what torch.amp.GradScaler hands over: the scale's inverse and the overflow flag
        kw["grad_scale"] = torch.full((1,), 1.0 / 1024.0, device=device)
        kw["found_inf"] = torch.zeros(1, device=device)
    outputs = [p_flat.all]
    for step in range(2):
        _gradient(g_flat.all, gen, kind)
        if unseen is not None:
            params[0].grad[unseen] = 0.0
        if case["amp"]:
            g_flat.all.mul_(1024.0)
        opt.step(**kw)
        if step == 0:
            outputs += _lay_flat(opt, params)
    return {"opt": opt, "kw": kw, "out": outputs, "clip": case["clip"]}


def _lay_flat(opt, params):
    """Moves every kind of state tensor into a flat buffer of its own; returns the buffers."""
    places = {}      # (name, dtype) -> [(holder, key, tensor)]
    for p in params:
        st = opt.state[p]
        for key in ("exp_avg", "exp_avg_sq"):
            places.setdefault((key, st[key].dtype), []).append((st, key, st[key]))
        for name in ("momentum_qstate", "variance_qstate"):
            over = st[name]["overhead"]
            if torch.is_tensor(over.get("max1")):
                places.setdefault((name, torch.float32), []).append((over, "max1", over["max1"]))
            for d, t in enumerate(over.get("max_dims") or ()):
                places.setdefault(("max_dims", torch.float32), []).append((over["max_dims"], d, t))
    buffers = []
    for (_, dtype), items in places.items():
        flat = _Flat([t.numel() for _, _, t in items], dtype, params[0].device)
        for view, (holder, key, t) in zip(flat.views, items):
            holder[key] = view.view(t.shape).copy_(t)
        buffers.append(flat.all)
    return buffers


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=device).manual_seed(seed)
    if case["do"] == "step":
        return _prepare_step(case, gen, device) | {"do": "step"}
    if case["do"] == "call":
        n = case["numel"]
        p = torch.empty(n, dtype=DTYPES[case["p"]], device=device)
        g = torch.empty(n, dtype=DTYPES[case["g"]], device=device)
        _normal(p, gen, 0.02)
        zeros = lambda k, dt: torch.zeros(k, dtype=dt, device=device)
        if n > THRESHOLD:
            nbytes, nblk = state_sizes(n)
            state = [zeros(nbytes, torch.uint8), zeros(nbytes, torch.uint8), zeros(nblk, torch.float32), zeros(nblk, torch.float32)]
        else:
            state = [zeros(n, torch.float32), zeros(n, torch.float32)]
        s = {"do": "call", "p": p, "g": g, "state": state, "step": 0}
        for _ in range(2):
            _gradient(g, gen, "outliers")
            run(s)
        return s
    rows, cols = case["rows"], case["cols"]
    m = torch.empty(rows, cols, device=device)
    v = torch.empty(rows, cols, device=device)
    _gradient(m.view(-1), gen, "heavy")
    _gradient(v.view(-1), gen, "heavy")
    v.square_()
    s = {"do": case["do"], "scale": case["scale"], "m": m, "v": v}
    if case["do"] == "decode":
        s["packed"] = _encode(s)
        del s["m"], s["v"]
        s["numel"] = rows * cols
    return s


def _encode(s):
    if s["scale"] == "rank1":
        return (*quantize_state(s["m"], 0), *quantfour_hip.quantize_state_rank1(s["v"]))
    return (*quantize_state(s["m"], 0), *quantize_state(s["v"], 1))


# -- one pass -----------------------------------------------------------------
def run(state):
    if state["do"] == "step":
        state["opt"].step(**state["kw"])
        return [*state["out"], state["opt"].last_grad_norm] if state["clip"] else state["out"]
    if state["do"] == "call":
        state["step"] += 1
        call = fused_4bit if len(state["state"]) == 4 else fused_single_tensor
        call(state["p"], state["g"], *state["state"], HP["betas"][0], HP["betas"][1], HP["lr"], HP["weight_decay"],
             HP["eps"], state["step"])
        return [state["p"], *state["state"]]
    if state["do"] == "encode":
        return _encode(state)
    m_codes, m_scales, v_codes, *v_scales = state["packed"]
    m = dequantize_state(m_codes, m_scales, state["numel"], 0)
    if state["scale"] == "rank1":
        return m, quantfour_hip.dequantize_state_rank1(v_codes, *v_scales)
    return m, dequantize_state(v_codes, v_scales[0], state["numel"], 1)


# -- what a pass cannot do without ---------------------------------------------
def work(case):
    """Every input read once, every output written once (a clipped step reads its gradients
    once here, though their norm has to be known before the first use; likewise rank-1 scaling
    and its maxima).  Operations: about thirty per element in a step."""
    block = 4.0 / 128
    if case["do"] in ("encode", "decode"):
        n = case["rows"] * case["cols"]
        second = block * n if case["scale"] == "group" else 4 * (case["rows"] + case["cols"])
        return {"bytes": n * (2 * 4.5 + block) + second, "flops": 4 * n}
    if case["do"] == "call":
        sizes, shapes = [case["numel"]], [(case["numel"],)]
    else:
        shapes = shapes_of(case)
        sizes = [_numel(s) for s in shapes]
    total = 0.0
    for n, shape in zip(sizes, shapes):
        total += n * (2 * SIZE[case["p"]] + SIZE[case["g"]])
        if n <= THRESHOLD:
            total += 16 * n
        elif case.get("scale") == "rank1" and 2 <= len(shape) and shape[-1] >= 2:
            total += n * (2 + 2 * block) + 8 * sum(shape)
        else:
            total += n * (2 + 4 * block)
    return {"bytes": total, "flops": 30.0 * sum(sizes)}


def tolerance(case):
    """Codes, scales and statistics are the same bytes for any correct implementation, and so
    are fp32 parameters with block scales and nearest rounding (the reference's expression,
    every operation rounded as IEEE 754 rounds it).  Elsewhere the parameter update is free to
    fold its constants and to use the hardware's square root and reciprocal: fp32 parameters
    move by parts in 1e7 of a step, 16-bit ones by one unit in the last place now and then.
    A clipped step multiplies by a coefficient from the fp32 norm, which may round to a
    neighbour when its sum is taken in another order: a code next to a threshold may flip."""
    # four times what was measured: the exact against the folded update (bf16 4.2e-6 and one
    # unit in the last place, 7.6e-3; fp32 1.4e-8 and 2.4e-7), a norm one unit in the last
    # place up (5.5e-6, 1.9e-2, 1.2e-6 of the codes)
    if case.get("clip"):
        return {"rel": 2e-5, "max": 0.08, "differ": 5e-6}
    if case["do"] in ("encode", "decode"):
        return "exact"
    if case["p"] != "float32":
        return {"rel": 2e-5, "max": 0.03}
    if case["do"] == "step" and (case["scale"] != "group" or case["round"] != "real-nearest"):
        return {"rel": 6e-8, "max": 1e-6}
    return "exact"
