"""The workloads this framework's speed is measured on.

A Muon program calls the framework in four ways, and each is here over the
sizes it is used at, from a single small weight to a whole transformer block:
the optimizer step itself (``torch.optim.Muon.step`` over the patched HIP path,
with plain and with chunked weights), the Newton–Schulz function alone (one
matrix, a batch), the AdamW half of the optimizer pair, and the two elementwise
ops that a program with its own loop calls around Newton–Schulz.

Every case is a dict of plain values:

``kind``
    ``ns``       newton_schulz of a [batch, rows, cols] input
    ``batched``  batched_gram_newtonschulz of a [batch, 128, cols] input
    ``step``     Muon step over ``count`` weights of rows x cols, each one
                 orthogonalised as ``chunks`` row blocks
    ``block``    Muon step over ``layers`` MMDiT blocks of width ``hidden``
    ``adamw``    AdamW step over the params Muon leaves to it in ``layers``
                 joint blocks of width ``hidden``
    ``ops``      muon_momentum_nesterov, then step_param, on a rows x cols weight
``dtype``
    ``f32``: params, grads and state in float32 (float32 masters); ``bf16``:
    params and grads in bfloat16, Muon's momentum in float32.
``form``
    the Newton–Schulz organisation, ``gram`` (the default) or ``standard``.
"""
from __future__ import annotations

import math

import torch

from pan2_amd.optim import kernels, patch_muon as pm
from pan2_amd.optim.patch_adamw import patch_adamw

DEVICE = "cuda:0"
COEFFS = (3.4445, -4.7750, 2.0315)
STEPS, EPS = 5, 1e-7
MU, LR, WD = 0.95, 0.02, 0.01
ADJUST = "match_rms_adamw"
ADAM_LR, ADAM_BETA, ADAM_EPS, ADAM_WD = 1e-4, 0.95, 1e-8, 0.05
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # one narrow weight (a head of 96, a LoRA factor): launches and latency only
        dict(name="ns_96x320", kind="ns", batch=1, rows=96, cols=320, dtype="f32", form="gram"),
        # a small model's whole step, 30 weights of width 256 (the sizes the tests train at)
        dict(name="step_small_model", kind="block", hidden=256, layers=2, text=200, dtype="f32", form="gram"),
        # the benchmark's first configuration: one lone float32 1024 x 4096 weight
        dict(name="step_1024x4096", kind="step", rows=1024, cols=4096, count=1, chunks=1, dtype="f32",
             form="standard"),
        # a few weights whose sides divide by nothing
        dict(name="step_777x1900", kind="step", rows=777, cols=1900, count=3, chunks=1, dtype="bf16", form="gram"),
        # one block of a mid-size model, mixed wide, tall and square weights
        dict(name="step_block_1024", kind="block", hidden=1024, layers=1, text=1000, dtype="bf16", form="gram"),
        # one attention projection of the large model on its own, as torch's own function computes it
        dict(name="ns_2048x2048", kind="ns", batch=1, rows=2048, cols=2048, dtype="bf16", form="standard"),
        # some of the benchmark's 5120 x 5120 attention projections, float32 masters
        dict(name="step_5120x5120", kind="step", rows=5120, cols=5120, count=4, chunks=1, dtype="f32",
             form="standard"),
        # one dual-stream MMDiT block at full width, the benchmark's unit; the largest case
        dict(name="step_mmdit_block", kind="block", hidden=5120, layers=1, text=4096, dtype="bf16", form="gram"),
        # one joint block's QKV weight, 192 row blocks of 128 x 4096, torch's quintic
        dict(name="step_qkv_192", kind="step", rows=24576, cols=4096, count=1, chunks=192, dtype="f32",
             form="standard"),
        # four of them in the default form (drawn cases also run such batches of
        # 128-row blocks through batched_gram_newtonschulz, without the step)
        dict(name="step_qkv_768", kind="step", rows=24576, cols=4096, count=4, chunks=192, dtype="bf16",
             form="gram"),
        # the AdamW half over a full model's biases, norms, embedders and head
        dict(name="adamw_44_layers", kind="adamw", hidden=4096, layers=44, dtype="f32"),
        # momentum and param step of one 5120 x 4096 weight, for a program that runs its own loop
        dict(name="ops_5120x4096", kind="ops", rows=5120, cols=4096, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    largest = work(next(c for c in listed() if c["name"] == "step_mmdit_block"))
    while True:
        kind = rng.choice(("ns", "step", "step", "block", "chunks", "batched", "adamw", "ops"))
        dtype, form = rng.choice(("f32", "bf16")), rng.choice(("gram", "standard"))
        if kind == "ns":
            case = dict(kind="ns", batch=rng.choice((1, 1, 2, 5)), rows=_log(rng, 16, 4096), cols=_log(rng, 16, 4096),
                        dtype=dtype, form=form)
        elif kind == "step":
            case = dict(kind="step", rows=_log(rng, 64, 6144), cols=_log(rng, 64, 6144), count=_log(rng, 1, 8),
                        chunks=1, dtype=dtype, form=form)
        elif kind == "block":
            case = dict(kind="block", hidden=_log(rng, 128, 2048), layers=rng.choice((1, 2)),
                        text=_log(rng, 100, 2000), dtype=dtype, form=form)
        elif kind == "chunks":
            chunks = _log(rng, 12, 192)
            case = dict(kind="step", rows=128 * chunks, cols=_log(rng, 256, 4096), count=_log(rng, 1, 6),
                        chunks=chunks, dtype=dtype, form=form)
        elif kind == "batched":
            case = dict(kind="batched", batch=_log(rng, 96, 512), cols=_log(rng, 128, 6144), dtype="bf16", form="gram")
        elif kind == "adamw":
            case = dict(kind="adamw", hidden=_log(rng, 64, 4096), layers=_log(rng, 1, 44), dtype=dtype)
        else:
            case = dict(kind="ops", rows=_log(rng, 16, 8192), cols=_log(rng, 16, 8192), dtype=dtype)
        w = work(case)
        if w["flops"] <= largest["flops"] and w["bytes"] <= largest["bytes"]:
            return case


# ---------------------------------------------------------------- shapes


def _weights(case):
    """Shapes of the Muon weights of a step."""
    if case["kind"] == "step":
        return [(case["rows"], case["cols"])] * case["count"]
    h, t = case["hidden"], case["text"]
    return ([(h, h)] * 8 + [(4 * h, h)] * 2 + [(h, 4 * h)] * 2 + [(h, 6 * h)] * 2 + [(t, h)]) * case["layers"]


def _matrices(case):
    """Shapes that Newton–Schulz runs on."""
    if case["kind"] == "ns":
        return [(case["rows"], case["cols"])] * case["batch"]
    if case["kind"] == "batched":
        return [(128, case["cols"])] * case["batch"]
    n = case.get("chunks", 1)
    return [(r // n, c) for r, c in _weights(case) for _ in range(n)]


def _adamw_shapes(case):
    """Biases, norm weights and modulation vectors of the blocks, then the
    embedders and the head."""
    h = case["hidden"]
    block = [(6 * h,), (2 * h,), (8 * h,), (h,), (4 * h,), (h,), (256,), (256,), (6 * h,)]
    ends = [(3, h), (h,), (h, h), (h,), (h, 256), (h,), (h, h), (h,), (h, 64), (h,), (64, h), (64,), (2 * h, h),
            (2 * h,)]
    return block * case["layers"] + ends


def _ns_flops(shape, form):
    """Products Newton–Schulz cannot do without, symmetric ones counted once."""
    m, n = min(shape), max(shape)
    gram, square, apply = m * (m + 1) * n, m * m * (m + 1), 2 * m * m * n
    if form == "standard":
        return STEPS * (gram + square + apply)
    # two segments (iterations 0-1 and 2-4): a gram and an application each;
    # Z every iteration, Q after a segment's first, R Z and Z R Z unless the
    # segment ends
    return 2 * (gram + apply) + (5 + 3 + 2 * 3) * square


def work(case):
    kind = case["kind"]
    wide = case["dtype"] == "f32"
    if kind == "adamw":
        # param, exp_avg, exp_avg_sq read and written, grad read
        return {"bytes": (28 if wide else 14) * sum(math.prod(s) for s in _adamw_shapes(case)), "flops": 0}
    if kind == "ops":
        n = case["rows"] * case["cols"]
        # grad read, momentum read and written, update written and read, param read and written
        return {"bytes": n * (28 if wide else 18), "flops": 0}
    mats = _matrices(case)
    flops = sum(_ns_flops(s, case["form"]) for s in mats)
    n = sum(r * c for r, c in mats)
    if kind in ("ns", "batched"):
        return {"bytes": n * ((4 if wide else 2) + 2), "flops": flops}
    # grad read, momentum read and written, param read and written
    return {"bytes": n * (20 if wide else 14), "flops": flops}


def tolerance(case):
    # about four times the distance to exact() measured over some 80 cases
    if case["kind"] in ("adamw", "ops"):
        return {"rel": 3e-7 if case["dtype"] == "f32" else 8e-3}  # one rounding of each result
    gram = case["form"] == "gram"
    if case["kind"] in ("ns", "batched"):
        # 0.9% to 1.8% from bf16 products; the gram form reaches 4.5% on square
        # inputs, whose smallest singular values it resolves least
        m, n = min(_matrices(case)[0]), max(_matrices(case)[0])
        return {"rel": 0.16 if gram and 2 * n < 3 * m else 0.07}
    # the same, seen through the params: a step moves them by about a fifth of their size
    return {"rel": 4e-2 if gram else 1.2e-2}


# ---------------------------------------------------------------- inputs


def _grad(shape, dtype, gen):
    """A gradient: Gaussian entries, rows of different scale."""
    g = torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(0.0, 1e-3, generator=gen)
    if len(shape) > 1:
        scale = torch.empty((*shape[:-1], 1), dtype=torch.float32, device=DEVICE).normal_(0.0, 0.3, generator=gen)
        g.mul_(scale.exp_())
    return g.to(dtype)


def _weight(shape, dtype, gen):
    return torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(0.0, 0.02, generator=gen).to(dtype)


def _flat(shapes, dtype):
    """One buffer that holds tensors of these shapes, and the tensors (each at a
    256-byte boundary, as an allocator places it)."""
    starts, end = [], 0
    for s in shapes:
        starts.append(end)
        end += -(-math.prod(s) // 128) * 128
    buf = torch.zeros(end, dtype=dtype, device=DEVICE)
    return buf, [buf[o:o + math.prod(s)].view(s) for o, s in zip(starts, shapes)]


def _inputs(case, seed):
    """The tensors of a call, one list per role, from the seed alone."""
    gen = torch.Generator(DEVICE).manual_seed(seed)
    dt, kind = DTYPES[case["dtype"]], case["kind"]
    if kind == "ns":
        shape = (case["rows"], case["cols"])
        return {"x": [_grad((case["batch"], *shape) if case["batch"] > 1 else shape, dt, gen)]}
    if kind == "batched":
        return {"x": [_grad((case["batch"], 128, case["cols"]), dt, gen)]}
    if kind == "adamw":
        # the params and each part of their state lie in one buffer: a few
        # hundred small tensors, returned as three
        shapes = _adamw_shapes(case)
        data = {"g": [_grad(s, dt, gen) for s in shapes]}
        make = {"p": lambda s: _weight(s, dt, gen), "m": lambda s: 0.5 * _grad(s, dt, gen),
                "v": lambda s: torch.square(_grad(s, dt, gen)) + 1e-8}
        for k, f in make.items():
            data["flat_" + k], data[k] = _flat(shapes, dt)
            for t in data[k]:
                t.copy_(f(t.shape))
        return data
    shapes = _weights(case) if kind != "ops" else [(case["rows"], case["cols"])]
    return {"p": [_weight(s, dt, gen) for s in shapes], "g": [_grad(s, dt, gen) for s in shapes],
            "m": [_grad(s, torch.float32, gen) for s in shapes]}


def prepare(case, seed):
    data = _inputs(case, seed)
    state = dict(data, case=case)
    kind = case["kind"]
    if kind == "batched":
        # the op returns the result in its input's storage, as a step's update
        # buffer is used: each pass starts from the same update
        state["buf"] = torch.empty_like(data["x"][0])
    elif kind == "adamw":
        patch_adamw()
        params = _parameters(data)
        opt = torch.optim.AdamW(params, lr=torch.tensor(ADAM_LR, device=DEVICE), betas=(ADAM_BETA, ADAM_BETA),
                                eps=ADAM_EPS, weight_decay=ADAM_WD, fused=True)
        for p, m, v in zip(params, data["m"], data["v"]):
            opt.state[p].update(step=torch.tensor(9.0, device=DEVICE), exp_avg=m, exp_avg_sq=v)
        state["opt"] = opt
    elif kind in ("step", "block"):
        pm.patch_muon(case["form"])
        params = _parameters(data)
        group, n = {"params": params}, case.get("chunks", 1)
        if n > 1:
            group["adjust_lr_fn"] = (ADJUST, 0, n)  # as build_native_muon_optimizers writes its chunked groups
        opt = torch.optim.Muon([group], lr=torch.tensor(LR, device=DEVICE), weight_decay=WD, momentum=MU,
                               ns_coefficients=COEFFS, ns_steps=STEPS, eps=EPS, adjust_lr_fn=ADJUST)
        for p, m in zip(params, data["m"]):
            opt.state[p]["momentum_buffer"] = m
        state["opt"] = opt
    elif kind == "ops":
        state["lr"] = torch.tensor(LR, device=DEVICE)
    return state


def _parameters(data):
    params = [torch.nn.Parameter(p) for p in data["p"]]
    for p, g in zip(params, data["g"]):
        p.grad = g
    return params


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ns":
        pm.NS_FORM = case["form"]  # a program chooses the form once; here cases of both share a process
        return pm.newton_schulz(state["x"][0], COEFFS, STEPS, EPS)
    if kind == "batched":
        state["buf"].copy_(state["x"][0])
        return kernels.batched_gram_newtonschulz(state["buf"], (COEFFS,) * STEPS, STEPS, EPS)
    if kind == "adamw":
        state["opt"].step()
        return {k: state["flat_" + k] for k in "pmv"}
    if kind == "ops":
        p, g, m = state["p"][0], state["g"][0], state["m"][0]
        u = kernels.muon_momentum_nesterov(m, g, MU)
        kernels.step_param(p, u, state["lr"], WD, ADJUST, p.shape)
        return {"p": p, "m": m, "u": u}
    pm.NS_FORM = case["form"]
    state["opt"].step()
    return {"p": state["p"], "m": state["m"]}


# ---------------------------------------------------------------- in 64 bits


def _ns_exact(x):
    """The quintic iteration in float64 (both forms are this polynomial)."""
    a, b, c = COEFFS
    x = x.double()
    tall = x.shape[-2] > x.shape[-1]
    if tall:
        x = x.mT.contiguous()
    x = x / x.norm().clamp(min=EPS)
    for _ in range(STEPS):
        r = x @ x.T
        x = a * x + (b * r + c * (r @ r)) @ x
    return x.mT.contiguous() if tall else x


def _blocks(t, n):
    return [t[i * (t.shape[0] // n):(i + 1) * (t.shape[0] // n)] for i in range(n)]


def _ratio(shape):
    return 0.2 * math.sqrt(max(shape))


def exact(case, seed):
    data = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("ns", "batched"):
        x = data["x"][0]
        return _ns_exact(x) if x.ndim == 2 else torch.stack([_ns_exact(y) for y in x])
    if kind == "adamw":
        p, m, v = (data["flat_" + k].double() for k in "pmv")
        g, parts = _flat(_adamw_shapes(case), torch.float64)
        for t, s in zip(parts, data["g"]):
            t.copy_(s)
        fix = 1.0 - ADAM_BETA ** 10
        m.lerp_(g, 1.0 - ADAM_BETA)
        v.mul_(ADAM_BETA).addcmul_(g, g, value=1.0 - ADAM_BETA)
        p.mul_(1.0 - ADAM_LR * ADAM_WD).addcdiv_(m, (v / fix).sqrt_().add_(ADAM_EPS), value=-ADAM_LR / fix)
        return {"p": p, "m": m, "v": v}
    p, g, m = ([t.double() for t in data.pop(k)] for k in ("p", "g", "m"))
    for mi, gi in zip(m, g):
        mi.lerp_(gi, 1.0 - MU)
    u = [gi * (1.0 - MU) + mi * MU for gi, mi in zip(g, m)]
    del g
    if kind == "ops":
        p[0].mul_(1.0 - LR * WD).add_(u[0], alpha=-LR * _ratio(p[0].shape))
        return {"p": p[0], "m": m[0], "u": u[0]}
    for pi, ui in zip(p, u):
        for pb, ub in zip(_blocks(pi, case.get("chunks", 1)), _blocks(ui, case.get("chunks", 1))):
            pb.mul_(1.0 - LR * WD).add_(_ns_exact(ub), alpha=-LR * _ratio(pb.shape))
    return {"p": p, "m": m}
