"""Timed cases of the gradient-accumulation boundary, through the engine's API.

A case is a model's tensor list (``list``, ``layers``, ``width``, ``vocab``,
``context``, ``lead``), a precision and a way of taking the step (``path``):

``step``    the boundary of an ordinary training loop: the window's last
            backward left a gradient on every parameter, then
            ``engine.step()``.  At ZeRO stage 3 the forward's parameter
            gather comes first.
``window``  contiguous gradients: the gradient hooks of ``micro`` backward
            passes, their end-of-backward flushes, then ``engine.step()``.
``pieces``  the unfused step, call by call (flatten, overflow test, unscale,
            reduce, clip, Adam, sync), as a custom loop drives it.

Everything a pass changes comes back: masters, both moments, the model copy,
the gradient norm (and the flat gradient where the path exposes it).
"""

from __future__ import annotations

import math

import torch
from torch import nn

import minispeed_amd as ms
from minispeed_amd import precision
from minispeed_amd.workloads import gpt_shapes

LR, BETAS, EPS, DECAY, CLIP = 1e-4, (0.9, 0.999), 1e-8, 0.01, 1.0
STEPS_DONE = 100           # the state is that of a run under way
LOSS_SCALE_POWER = 16
GRAD_STD = 1e-3
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
ALIGN = 512                # bytes: where torch's allocator starts a tensor

_CASE = {"path": "step", "list": "gpt", "layers": 12, "width": 768, "vocab": 50257,
         "context": 1024, "lead": 0, "dtype": "fp16", "stage": 1, "groups": 1, "clip": True,
         "materialize": False, "micro": 1}


def _case(**kw):
    return {**_CASE, **kw}


def listed():
    gpt_350m = dict(layers=24, width=1024, vocab=50257, context=1024)
    return [
        # the smallest: a GPT for debugging or a unit test on the card; its
        # state fits the cache, so launches and host work count
        _case(name="step_tiny_lm_fp16", layers=4, width=256, vocab=512, context=128),
        # a convolutional net of odd width: hundreds of tensors, none of
        # them a multiple of any vector or tile, no clipping
        _case(name="step_conv_odd_bf16", list="conv", layers=48, width=151, dtype="bf16", stage=0,
              clip=False),
        # GPT-2 small, the ordinary single-GPU run
        _case(name="step_gpt2_124m_fp16", stage=2),
        # the same in full precision, behind a tensor of 3 elements (an
        # odd-sized bias): every later tensor off the flat space's grid
        _case(name="step_gpt2_124m_shift_fp32", lead=3, dtype="fp32"),
        # 350M in bf16, weights decayed and biases and norms not (the usual
        # two parameter groups)
        _case(name="step_350m_bf16_2groups", dtype="bf16", groups=2, **gpt_350m),
        # the fp32 flat gradient written as well (a user who inspects it)
        _case(name="step_350m_fp16_flat", materialize=True, **gpt_350m),
        # ZeRO-3: the forward's gather, then the boundary
        _case(name="gather_step_350m_bf16", dtype="bf16", stage=3, **gpt_350m),
        # contiguous gradients over a window of two micro-batches
        _case(name="window_124m_bf16", path="window", micro=2, dtype="bf16", stage=2),
        # the same over the odd convolutional net, four micro-batches
        _case(name="window_conv_odd_fp16", path="window", micro=4, list="conv", layers=48,
              width=151),
        # the step driven call by call
        _case(name="pieces_124m_fp16", path="pieces"),
        # the largest: 1.3B parameters on one GPU
        _case(name="step_1p3b_fp16", layers=24, width=2048, vocab=50257, context=2048),
    ]


def _shapes(case):
    if case["list"] == "gpt":
        body = gpt_shapes(case["layers"], case["width"], case["vocab"], case["context"])
    else:   # conv + bias + two norm vectors per layer
        c = case["width"]
        body = [s for _ in range(case["layers"]) for s in ((c, c, 3, 3), (c,), (c,), (c,))]
    return ([(case["lead"],)] if case["lead"] else []) + body


def _groups(case):
    """Shapes of each parameter group: one, or matrices and vectors apart."""
    shapes = _shapes(case)
    if case["groups"] == 1:
        return [shapes]
    return [[s for s in shapes if len(s) > 1], [s for s in shapes if len(s) == 1]]


def _numel(shapes):
    return sum(math.prod(s) for s in shapes)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    limit = work(listed()[-1])["bytes"]
    while True:
        kind = rng.choice(["gpt", "gpt", "gpt", "conv"])
        want = math.exp(rng.uniform(math.log(1e5), math.log(1.2e9 if kind == "gpt" else 1e8)))
        layers = _log_int(rng, 2, 48)
        width = max(24, int(math.sqrt(want / ((12 if kind == "gpt" else 9) * layers))))
        step = rng.choice([1, 1, 8, 64])
        width = max(step, width // step * step)
        case = _case(
            path=rng.choice(["step", "step", "step", "window", "pieces"]), list=kind, layers=layers,
            width=width, vocab=_log_int(rng, 64, 50257), context=_log_int(rng, 32, 2048),
            lead=rng.choice([0, 0, 0, 1, 3]), dtype=rng.choice(["fp16", "bf16", "bf16", "fp32"]),
            groups=rng.choice([1, 1, 2]), clip=rng.random() < 0.75)
        case["stage"] = rng.choice([0, 1, 2, 3] if case["path"] == "step" else [0, 1, 2])
        case["materialize"] = case["path"] == "step" and rng.random() < 0.2
        case["micro"] = rng.choice([1, 2, 4]) if case["path"] == "window" else 1
        n = _numel(_shapes(case))
        if 5e4 <= n and work(case)["bytes"] <= limit and width <= 2560:
            return case


# ------------------------------------------------------------------ inputs
def _padded(shapes, itemsize):
    """Start of every tensor, and the length, of a buffer that begins each
    tensor where the allocator would."""
    unit, at, starts = ALIGN // itemsize, 0, []
    for s in shapes:
        starts.append(at)
        at += -(-math.prod(s) // unit) * unit
    return starts, at


def _views(buf, shapes, starts):
    return [buf[o:o + math.prod(s)].view(s) for s, o in zip(shapes, starts)]


def _scale(case):
    return 2.0 ** LOSS_SCALE_POWER if case["dtype"] == "fp16" else 1.0


def _inputs(case, seed):
    """Per group: shapes, masters and moments (flat, in order) and one
    gradient buffer per micro-batch."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    out = []
    for shapes in _groups(case):
        n = _numel(shapes)

        def normal(k, std):
            return torch.empty(k, device="cuda").normal_(0.0, std, generator=gen)

        # typical of a run under way: |exp_avg| below sqrt(exp_avg_sq)
        state = normal(n, 0.02), normal(n, 3e-5), normal(n, 5e-5).add_(1e-4).square_()
        starts, size = _padded(shapes, dtype.itemsize)
        grads = [normal(size, GRAD_STD * _scale(case)).to(dtype) for _ in range(case["micro"])]
        out.append((shapes, state, starts, grads))
    return out


def _config(case):
    cfg = {
        "train_micro_batch_size_per_gpu": 1,
        "gradient_accumulation_steps": case["micro"],
        "gradient_clipping": CLIP if case["clip"] else None,
        "dtype": case["dtype"],
        "optimizer": {"type": "AdamW", "params": {"lr": LR, "betas": list(BETAS), "eps": EPS,
                                                  "weight_decay": DECAY}},
        "scheduler": {"type": "ConstantLR", "params": {"warmup_max_lr": LR}},
        "zero_optimization": {"stage": case["stage"]},
        "hip_boundary": {"materialize_flat_grad": case["materialize"],
                         "contiguous_gradients": case["path"] == "window"},
        "steps_per_print": 1000000,
    }
    if case["dtype"] == "fp16":
        cfg["fp16"] = {"enabled": True, "loss_scale": 0, "initial_scale_power": LOSS_SCALE_POWER,
                       "loss_scale_window": 1000}
    return cfg


class _State:
    """An engine mid-run and the gradients its backward passes left."""


def prepare(case, seed):
    groups = _inputs(case, seed)
    dtype = DTYPES[case["dtype"]]
    st = _State()
    st.case = case
    params, options = [], []
    for gi, (shapes, (master, _, _), _, _) in enumerate(groups):
        at, mine = 0, []
        for s in shapes:
            mine.append(nn.Parameter(master[at:at + math.prod(s)].view(s)))
            at += math.prod(s)
        params.append(mine)
        options.append({"params": mine, **({"weight_decay": 0.0} if gi else {})})
    st.engine = ms.initialize(model=nn.ParameterList([p for mine in params for p in mine]),
                              model_parameters=options, config=_config(case))
    st.params, st.grads, st.models = params, [], []
    for mine, (shapes, (_, m, v), starts, grads), flat, opt in zip(
            params, groups, st.engine.flat_groups, st.engine.optimizer.state):
        opt["exp_avg"].copy_(m)
        opt["exp_avg_sq"].copy_(v)
        opt["step"] = STEPS_DONE
        st.grads.append([_views(g, shapes, starts) for g in grads])
        if case["stage"] == 3:
            st.models.append(flat.model_shard)
            continue
        # the model's tensors in one buffer, each where an allocation of its
        # own would begin, so that the whole model copy is one output
        starts, size = _padded(shapes, dtype.itemsize)
        model = torch.zeros(size, dtype=dtype, device="cuda")
        for p, view in zip(mine, _views(model, shapes, starts)):
            p.data = view.copy_(p.data)
        st.models.append(model)
    return st


def _attach(st, micro):
    for mine, grads in zip(st.params, st.grads):
        for p, g in zip(mine, grads[micro]):
            p.grad = g


def run(st):
    case, engine = st.case, st.engine
    opt = engine.optimizer
    out = {}
    if case["path"] == "pieces":
        _attach(st, 0)
        for flat in engine.flat_groups:
            flat.flatten_grads()
        out["applied"] = not precision.has_overflow(*[flat.grad for flat in engine.flat_groups])
        for flat in engine.flat_groups:
            flat.unscale_grads(engine.loss_scale)
        opt.reduce_gradients()
        out["norm"] = opt.clip_gradients(engine.config.gradient_clipping)
        opt.step()
        opt.sync_parameters()
        out["grad"] = [flat.grad_for_shard() for flat in engine.flat_groups]
    else:
        if case["stage"] == 3:
            opt.gather_parameters()
        for micro in range(case["micro"]):
            _attach(st, micro)
            if case["path"] == "window":
                for gi, mine in enumerate(st.params):
                    for k, p in enumerate(mine):
                        engine.contiguous.accumulate(gi, k, p)
                engine.contiguous.flush()
            engine.micro_steps += 1
        out["applied"] = engine.step()
        out["norm"] = engine.get_gradient_norm()
    out["master"] = [flat.shard for flat in engine.flat_groups]
    out["exp_avg"] = [s["exp_avg"] for s in opt.state]
    out["exp_avg_sq"] = [s["exp_avg_sq"] for s in opt.state]
    out["model"] = st.models
    return out


# -------------------------------------------------------------------- work
def work(case):
    n, eb = _numel(_shapes(case)), DTYPES[case["dtype"]].itemsize
    if case["path"] == "pieces":
        # every call hands its result back before the next one: flatten
        # (eb + 4), overflow test 4, unscale 8, norm 4 and scaling 8, Adam
        # 28, sync (4 + eb)
        per = eb + 4 + 4 + 8 + (12 if case["clip"] else 4) + 28 + 4 + eb
    else:
        # masters and moments in and out, the model copy out, each
        # micro-batch's gradient in; the fp32 sums, or the flat gradient, out
        per = 24 + eb + eb * case["micro"]
        per += 4 if case["path"] == "window" or case["materialize"] else 0
        per += 4 + eb if case["stage"] == 3 else 0
    return {"bytes": per * n, "flops": (20 + 2 * case["micro"]) * n}


def tolerance(case):
    # Measured between two ways of writing the fp32 update (products fused
    # or not, the bias corrections folded or not, the norm one ulp apart):
    # masters and moments 5e-8 relative, 3e-7 at most; a model copy then
    # rounds the other way at a few elements, by one unit of its type
    # (2^-10, 2^-7), 3e-6 (fp16) and 1.1e-5 (bf16) relative.  Four times
    # that, and one unit.
    return {"fp32": {"rel": 2e-7, "max": 1.5e-6},
            "fp16": {"rel": 1.2e-5, "max": 1.1e-3},
            "bf16": {"rel": 4.5e-5, "max": 8.5e-3}}[case["dtype"]]


# ------------------------------------------------------------------- exact
def exact(case, seed):
    groups = _inputs(case, seed)
    grads = []
    for shapes, _, starts, micro in groups:
        total = None
        for buf in micro:
            g = torch.cat([v.reshape(-1).double() for v in _views(buf, shapes, starts)])
            total = g if total is None else total.add_(g)
        grads.append(total.div_(_scale(case)))
    norm = math.sqrt(sum(float(g.square().sum()) for g in grads))
    if case["clip"] and norm > CLIP:
        for g in grads:
            g.mul_(CLIP / (norm + 1e-6))
    out = {"applied": True, "norm": norm, "master": [], "exp_avg": [], "exp_avg_sq": [], "model": []}
    if case["path"] == "pieces":
        out["grad"] = grads
    step = STEPS_DONE + 1
    for gi, ((shapes, (p, m, v), _, _), g) in enumerate(zip(groups, grads)):
        p, m, v = (t.double() for t in (p, m, v))
        p.mul_(1.0 - LR * (0.0 if gi else DECAY))
        m.mul_(BETAS[0]).add_(g, alpha=1.0 - BETAS[0])
        v.mul_(BETAS[1]).addcmul_(g, g, value=1.0 - BETAS[1])
        den = (v / (1.0 - BETAS[1] ** step)).sqrt_().add_(EPS)
        p.addcdiv_(m, den, value=-LR / (1.0 - BETAS[0] ** step))
        out["master"].append(p)
        out["exp_avg"].append(m)
        out["exp_avg_sq"].append(v)
        if case["stage"] == 3:
            out["model"].append(p)
            continue
        starts, size = _padded(shapes, DTYPES[case["dtype"]].itemsize)
        model = torch.zeros(size, dtype=torch.float64, device="cuda")
        at = 0
        for s, o in zip(shapes, starts):
            model[o:o + math.prod(s)] = p[at:at + math.prod(s)]
            at += math.prod(s)
        out["model"].append(model)
    return out
