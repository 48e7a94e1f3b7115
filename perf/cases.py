"""What a training program asks of this package, as cases that can be timed.

A case is one optimizer step as a user's loop makes it, through ``LayerAdam``'s
public methods, on moments warmed by earlier steps:

``flat``     a layer held flat in HBM: optional clip, then one ``step_chunk`` that
             also writes the bf16 compute copy;
``tensors``  a layer of separate parameters in HBM: optional clip over the list of
             grads, then ``step(layer)`` (grads in ``p.grad``) or
             ``step_with_grad_views`` (a dict of views into a flat grad buffer);
``stack``    a whole small model in HBM, in sliding order: the global norm is
             accumulated layer by layer, then every layer is stepped;
``host``     a layer whose state stays in host RAM, stepped in the runtime's
             32 Mi-element ``step_chunk`` calls;
``host_tensors``  a layer of separate host parameters, ``step(layer)``.
"""
import math

import torch

from slideformer_amd import LayerAdam

DEVICE = "cuda:0"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZES = {"f32": 4, "bf16": 2, "f16": 2}
STEP = 5            # steps taken before: the moments are warm
LR, BETAS, EPS = 1e-5, (0.9, 0.999), 1e-8
CALL_ELEMS = 32 * 1024 * 1024   # the runtime's elements per step_chunk call


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _flat(n, dtypes="f32/bf16/f32", clip=True, wd=0.01, off=0, outliers=False):
    return {"kind": "flat", "n": n, "dtypes": dtypes, "clip": clip, "wd": wd, "off": off, "outliers": outliers}


def _tensors(family, hidden, ffn, kv, dtypes, views, clip):
    return {"kind": "tensors", "family": family, "hidden": hidden, "ffn": ffn, "kv": kv, "dtypes": dtypes,
            "views": views, "clip": clip}


def _host(n, master, moments, overlap):
    return {"kind": "host", "n": n, "master": master, "moments": moments, "overlap": overlap}


def listed():
    return [
        # The smallest layer of a model that is stepped layer by layer: its final norm of 4096 scales.
        dict(_flat(4096), name="final_norm_flat"),
        # One GPT-2-small block held flat, clipped over itself: an ordinary small layer.
        dict(_flat(7_087_872), name="gpt2_block_flat"),
        # One Llama-3.1-8B decoder layer held flat with its state in HBM: the flagship step.
        dict(_flat(218_112_000), name="llama8b_layer_flat"),
        # One rank's seventh of a Qwen2.5-14B layer: an odd number of elements, own master and moments, the grads
        # and the compute copy at the rank's place in the layer's buffers; a few large grads make the clip bite.
        dict(_flat(39_324_087, wd=0.1, off=39_324_087, outliers=True), name="qwen14b_layer_shard"),
        # The twelve parameters of a GPT-2-small block, grads as views of the runtime's flat grad buffer.
        dict(_tensors("gpt2", 768, 3072, 768, "f32/bf16/f32", True, True), name="gpt2_block_tensors"),
        # The nine parameters of a Llama-3.1-8B layer trained in bf16 with bf16 moments (fp32_optimizer_state=False).
        dict(_tensors("llama", 4096, 14336, 1024, "bf16/bf16/bf16", False, False), name="llama8b_layer_bf16"),
        # A block of odd width trained in bf16 with fp32 moments: every parameter its own tensor, the moments slices
        # of the layer's flat buffers, so most of them start at different places of a 16-byte line.
        dict(_tensors("gpt2", 1023, 4092, 1023, "bf16/bf16/f32", False, True), name="odd_block_tensors"),
        # GPT-2 small whole: embedding and twelve blocks, one global clip in sliding order.
        {"kind": "stack", "layers": 12, "n": 7_087_872, "extra": 39_385_344, "name": "gpt2_model_stack"},
        # The runtime's own layout and calls: fp32 master and moments in pageable host RAM, page-locked grads.
        dict(_host(218_112_000, "pageable", "pageable", False), name="llama8b_layer_host"),
        # The moments in HBM beside a page-locked host master, calls that return once queued.
        dict(_host(218_112_000, "pinned", "hbm", True), name="llama8b_layer_hbm_moments"),
        # One GPT-2-small block in pageable host RAM: a host call of less than one chunk.
        dict(_host(7_087_872, "pageable", "pageable", False), name="gpt2_block_host"),
        # The twelve parameters of a GPT-2-small block on the host, grads in p.grad.
        {"kind": "host_tensors", "family": "gpt2", "hidden": 768, "ffn": 3072, "kv": 768, "name": "gpt2_block_host_tensors"},
    ]


def _log(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["flat", "flat", "flat", "tensors", "tensors", "tensors", "stack", "host", "host",
                       "host_tensors"])
    triples = ["f32/bf16/f32", "f32/bf16/f32", "f32/f32/f32", "bf16/bf16/f32", "bf16/bf16/bf16", "bf16/f32/f32",
               "f16/f16/f32", "f32/f16/f32", "f16/f32/f32"]
    if kind == "flat":
        n = _log(rng, 4096, 200_000_000)
        n = n | 1 if rng.random() < 0.4 else n // 64 * 64
        return _flat(n, rng.choice(triples), rng.random() < 0.6, rng.choice([0.0, 0.01, 0.1]),
                     rng.choice([0, 0, n]), rng.random() < 0.5)
    if kind == "tensors":
        family = rng.choice(["gpt2", "llama"])
        hidden = _log(rng, 64, 3500)
        hidden = hidden | 1 if rng.random() < 0.3 else max(64, hidden // 64 * 64)
        ffn = 4 * hidden if family == "gpt2" else int(hidden * 3.5)
        kv = hidden if family == "gpt2" else max(1, hidden // 4)
        return _tensors(family, hidden, ffn, kv, rng.choice(triples), rng.random() < 0.5, rng.random() < 0.6)
    if kind == "stack":
        h = max(64, _log(rng, 128, 1024) // 64 * 64)
        return {"kind": "stack", "layers": rng.randint(2, 12), "n": 12 * h * h + 13 * h,
                "extra": _log(rng, 1 << 20, 40_000_000)}
    if kind == "host":
        n = _log(rng, 65536, 200_000_000)
        n = n | 1 if rng.random() < 0.4 else n // 64 * 64
        return _host(n, rng.choice(["pageable", "pinned"]), rng.choice(["pageable", "pinned", "hbm"]),
                     rng.random() < 0.4)
    h = max(64, _log(rng, 128, 1600) // 64 * 64)
    return {"kind": "host_tensors", "family": "gpt2", "hidden": h, "ffn": 4 * h, "kv": h}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _shapes(c):
    h, f, kv = c["hidden"], c["ffn"], c["kv"]
    if c["family"] == "gpt2":
        return [(h,), (h,), (3 * h, h), (3 * h,), (h, h), (h,), (h,), (h,), (f, h), (f,), (h, f), (h,)]
    return [(h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f), (h,), (h,)]


def _count(shapes):
    return sum(math.prod(s) for s in shapes)


def _values(seed, n, dtypes, outliers=False, salt=0):
    """Master, grads and warm moments of n elements, on the GPU, in their own types."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed * 1009 + salt)
    pt, gt, st = (DTYPES[x] for x in dtypes.split("/"))

    def normal(std):
        return torch.randn(n, generator=gen, device=DEVICE).mul_(std)

    p = normal(0.02).to(pt)
    g = normal(1e-3)
    if outliers:
        g[torch.randint(n, (max(1, n // 1000),), generator=gen, device=DEVICE)] *= 100
    g = g.to(gt)
    m = normal(4e-4).to(st)
    v = normal(7e-5).square_().to(st)
    return p, g, m, v


def _adam(wd, **options):
    return LayerAdam(lr=LR, betas=BETAS, eps=EPS, weight_decay=wd, **options)


def _register(adam, idx, params, m, v):
    adam.add_layer_params(idx, params)
    adam.exp_avg_flat[idx].copy_(m)
    adam.exp_avg_sq_flat[idx].copy_(v)
    group = adam.param_groups[idx]
    group["step"] = STEP
    return group


def _prepare_flat(c, seed):
    n, off = c["n"], c["off"]
    p, g0, m, v = _values(seed, n, c["dtypes"], c["outliers"])
    adam = _adam(c["wd"], fp32_optimizer_state=m.dtype == torch.float32)
    _register(adam, 0, [torch.nn.Parameter(p, requires_grad=False)], m, v)
    g = torch.empty(off + n, dtype=g0.dtype, device=DEVICE)[off:].copy_(g0)
    out = torch.empty(off + n, dtype=torch.bfloat16, device=DEVICE)[off:]
    return {"case": c, "adam": adam, "p": p, "g": g, "out": out}


def _run_flat(s):
    adam = s["adam"]
    coef = norm = None
    if s["case"]["clip"]:
        coef, norm = adam.clip_grad_norm([s["g"]], 1.0)
    group = adam.begin_chunk_step(0)
    adam.step_chunk(s["p"], s["g"], adam.exp_avg_flat[0], adam.exp_avg_sq_flat[0], group, bf16_out=s["out"],
                    clip_coef=coef)
    adam.end_chunk_step(0)
    return {"p": s["p"], "m": adam.exp_avg_flat[0], "v": adam.exp_avg_sq_flat[0], "out": s["out"],
            "coef": coef, "norm": norm}


def _cut(flat, shapes, own):
    got, at = [], 0
    for shape in shapes:
        size = math.prod(shape)
        piece = flat[at:at + size].view(shape)
        got.append(piece.clone() if own else piece)
        at += size
    return got


def _prepare_tensors(c, seed):
    shapes = _shapes(c)
    p, g, m, v = _values(seed, _count(shapes), c["dtypes"])
    adam = _adam(0.01, fp32_optimizer_state=m.dtype == torch.float32)
    params = [torch.nn.Parameter(x, requires_grad=False) for x in _cut(p, shapes, not c["views"])]
    grads = _cut(g, shapes, not c["views"])
    _register(adam, 0, params, m, v)
    same = g.dtype == p.dtype
    if not c["views"] and same:
        for q, x in zip(params, grads):
            q.grad = x
    # p.grad has the parameter's type: grads of another type come as a dict, as the runtime's views do
    views = dict(zip(params, grads)) if c["views"] or not same else None
    return {"case": c, "adam": adam, "params": params, "grads": grads, "views": views}


def _run_tensors(s):
    adam = s["adam"]
    coef = norm = None
    if s["case"]["clip"]:
        coef, norm = adam.clip_grad_norm(s["grads"], 1.0)
    if s["views"] is not None:
        adam.step_with_grad_views(0, s["views"], clip_coef=coef)
    else:
        adam.step(0, clip_coef=coef)
    return {"p": s["params"], "m": adam.exp_avg_flat[0], "v": adam.exp_avg_sq_flat[0], "coef": coef, "norm": norm}


def _stack_sizes(c):
    return [c["extra"]] + [c["n"]] * c["layers"]


def _prepare_stack(c, seed):
    adam = _adam(0.01)
    layers = []
    for i, n in enumerate(_stack_sizes(c)):
        p, g, m, v = _values(seed, n, "f32/bf16/f32", salt=i + 1)
        _register(adam, i, [torch.nn.Parameter(p, requires_grad=False)], m, v)
        layers.append((p, g, torch.empty(n, dtype=torch.bfloat16, device=DEVICE)))
    return {"case": c, "adam": adam, "layers": layers}


def _run_stack(s):
    adam, layers = s["adam"], s["layers"]
    order = range(len(layers) - 1, -1, -1)
    norm_of = adam.grad_norm_begin(DEVICE)
    for i in order:
        norm_of.add(layers[i][1])
    coef, norm = norm_of.finish(1.0)
    for i in order:
        p, g, out = layers[i]
        group = adam.begin_chunk_step(i)
        adam.step_chunk(p, g, adam.exp_avg_flat[i], adam.exp_avg_sq_flat[i], group, bf16_out=out, clip_coef=coef)
        adam.end_chunk_step(i)
    return {"p": [x[0] for x in layers], "m": list(adam.exp_avg_flat.values()),
            "v": list(adam.exp_avg_sq_flat.values()), "out": [x[2] for x in layers], "coef": coef, "norm": norm}


def _to_host(x, pinned):
    return torch.empty(x.shape, dtype=x.dtype, pin_memory=pinned).copy_(x)


def _prepare_host(c, seed):
    p, g, m, v = _values(seed, c["n"], "f32/bf16/f32")
    adam = _adam(0.01, overlap_host_chunks=c["overlap"], pin_host_state=c["moments"] == "pinned",
                 moments_device=DEVICE if c["moments"] == "hbm" else None)
    master = _to_host(p, c["master"] == "pinned")
    _register(adam, 0, [torch.nn.Parameter(master, requires_grad=False)], m, v)
    return {"case": c, "adam": adam, "p": master, "g": _to_host(g, True),
            "out": torch.empty(c["n"], dtype=torch.bfloat16, device=DEVICE)}


def _run_host(s):
    adam, n = s["adam"], s["case"]["n"]
    m, v = adam.exp_avg_flat[0], adam.exp_avg_sq_flat[0]
    group = adam.begin_chunk_step(0)
    for a in range(0, n, CALL_ELEMS):
        b = min(n, a + CALL_ELEMS)
        adam.step_chunk(s["p"][a:b], s["g"][a:b], m[a:b], v[a:b], group, bf16_out=s["out"][a:b])
    adam.end_chunk_step(0)
    return {"p": s["p"], "m": m, "v": v, "out": s["out"]}


def _prepare_host_tensors(c, seed):
    shapes = _shapes(c)
    p, g, m, v = (x.cpu() for x in _values(seed, _count(shapes), "f32/f32/f32"))
    adam = _adam(0.01)
    params = [torch.nn.Parameter(x, requires_grad=False) for x in _cut(p, shapes, True)]
    _register(adam, 0, params, m, v)
    for q, x in zip(params, _cut(g, shapes, True)):
        q.grad = x
    return {"case": c, "adam": adam, "params": params}


def _run_host_tensors(s):
    adam = s["adam"]
    adam.step(0)
    return {"p": s["params"], "m": adam.exp_avg_flat[0], "v": adam.exp_avg_sq_flat[0]}


_PREPARE = {"flat": _prepare_flat, "tensors": _prepare_tensors, "stack": _prepare_stack, "host": _prepare_host,
            "host_tensors": _prepare_host_tensors}
_RUN = {"flat": _run_flat, "tensors": _run_tensors, "stack": _run_stack, "host": _run_host,
        "host_tensors": _run_host_tensors}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["case"]["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    dtypes, out = case.get("dtypes", "f32/bf16/f32"), True
    if kind == "tensors":
        n, out = _count(_shapes(case)), False
    elif kind == "host_tensors":
        n, out, dtypes = _count(_shapes(case)), False, "f32/f32/f32"
    else:
        n = sum(_stack_sizes(case)) if kind == "stack" else case["n"]
    p, g, s = (SIZES[x] for x in dtypes.split("/"))
    # 16: the multiplies, adds, root and quotient of one element
    return {"bytes": n * (2 * p + g + 4 * s + (2 if out else 0)), "flops": 16 * n}


def tolerance(case):
    # Without a clip every element is a fixed sequence of IEEE operations: the results are the reference CPU
    # Adam's, bit for bit.  With one, the norm is a float64 sum whose order is free, so the fp32 coefficient may
    # round the other way: one unit in the last place of the moments, and a bf16 rounding that goes the other way
    # here and there.
    # Seen with the coefficient moved by one unit: rel up to 8.3e-7, the largest difference 3.4e-3 (one bf16 unit).
    if case["kind"] == "stack" or case.get("clip"):
        return {"rel": 3.3e-6, "max": 1.4e-2}
    return "exact"


# ---------------------------------------------------------------------------
# the same step in 64 bits
# ---------------------------------------------------------------------------
def _f32(x):
    return float(torch.tensor(x, dtype=torch.float32))


def _exact_step(p, g, m, v, wd, coef):
    """The step on float64 values; the hyper-parameters are fp32, as the entry points take them."""
    t = STEP + 1
    b1, b2, lr, eps, wd = _f32(BETAS[0]), _f32(BETAS[1]), _f32(LR), _f32(EPS), _f32(wd)
    p, g, m, v = (x.double() for x in (p, g, m, v))
    g = g * coef if coef is not None else g
    m = m * b1 + g * (1 - b1)
    v = v * b2 + g * g * (1 - b2)
    u = (m / (1 - b1 ** t)) / (v.sqrt() / math.sqrt(1 - b2 ** t) + eps)
    return p - p * (lr * wd) - u * lr, m, v


def _exact_clip(grads):
    norm = sum(x.double().square().sum() for x in grads).sqrt().reshape(1)
    return torch.clamp(1.0 / (norm + 1e-6), max=1.0), norm


def exact(case, seed):
    kind = case["kind"]
    if kind == "stack":
        layers = [_values(seed, n, "f32/bf16/f32", salt=i + 1) for i, n in enumerate(_stack_sizes(case))]
        coef, norm = _exact_clip([x[1] for x in layers])
        got = [_exact_step(*x, 0.01, coef) for x in layers]
        return {"p": [x[0] for x in got], "m": [x[1] for x in got], "v": [x[2] for x in got],
                "out": [x[0] for x in got], "coef": coef, "norm": norm}
    if kind in ("flat", "host"):
        p, g, m, v = _values(seed, case["n"], case.get("dtypes", "f32/bf16/f32"), case.get("outliers", False))
        coef, norm = _exact_clip([g]) if case.get("clip") else (None, None)
        p, m, v = _exact_step(p, g, m, v, case.get("wd", 0.01), coef)
        got = {"p": p, "m": m, "v": v, "out": p}
        return got if kind == "host" else dict(got, coef=coef, norm=norm)
    shapes = _shapes(case)
    p, g, m, v = _values(seed, _count(shapes), case.get("dtypes", "f32/f32/f32"))
    coef, norm = _exact_clip([g]) if case.get("clip") else (None, None)
    p, m, v = _exact_step(p, g, m, v, 0.01, coef)
    got = {"p": _cut(p, shapes, False), "m": m, "v": v}
    return got if kind == "host_tensors" else dict(got, coef=coef, norm=norm)
