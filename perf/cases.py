"""The measured cases of the framework: what a training program has its optimizer store do.

Each case drives the public Python surface (`ttperf.ParamStore` and the optimizers) the way a
training loop does, on one GPU, with the store on torch's current stream:

  step      `opt.step()` on gradients that are in the store: the optimizer step alone
  backward  one iteration as a backward hands its gradients over: `opt.zero_grad()`, the
            gradients bucket by bucket (`accumulate_grads`, about 25 MB each, last layers first),
            for `micro` micro-batches, then `opt.step()`
  transfer  the optimizer state to contiguous device tensors (`download`) and another state back
            (`upload`), as checkpoints and weight averaging do

A case's plain values: the tensor table (`table` and its sizes), the store (`mode`, `layout`),
the optimizer (`opt`, `clip`, `scale`, `groups`) and what the pass does (`kind`, ...).
"""
import gc
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "tt-perf_amd"))
import ttperf  # noqa: E402
from ttperf import configs  # noqa: E402

LR, BETAS, EPS, WD = 6e-4, (0.9, 0.95), 1e-8, 0.1
SGD_LR, MOMENTUM = 0.1, 0.9
T0 = 1000  # steps already taken when a case starts (one optimizer per store)
BUCKET_BYTES = 25 << 20
BUCKET_TENSORS = 64
GRAD_STD, WEIGHT_STD = 1e-3, 0.02
MAX_PARAMS = 1_500_000_000  # of a drawn case

BASE = dict(kind="step", table="gpt", n_layer=12, d_model=768, vocab=50257, ctx=1024, shards=1,
            mode="mixed", layout="default", opt="adamw", clip=1.0, scale=0.0, groups=1,
            captured=False, source="bf16", micro=1, sums=False)


def _case(**kw):
    return {**BASE, **kw}


def listed():
    nano = dict(n_layer=6, d_model=384, vocab=65, ctx=256)
    large = dict(n_layer=36, d_model=1280)
    return [
        # the reference's example model: the smallest step, bound by launches and the host
        _case(name="mlp_adamw", table="mlp", d_in=64, d_hidden=128, d_out=10, mode="fp32"),
        # fine-tuning small odd-sized adapters with two learning rates: two optimizers over one
        # loss-scaled store, the second of which moves the scale
        _case(name="adapters_two_groups", table="ragged", n_tensors=300, mean_numel=4000,
              scale=65536.0, groups=2),
        # nanoGPT's character model: the small-model step
        _case(name="nanogpt_char_adamw", **nano),
        # one GPU's ZeRO-1 shard (of 8) of GPT-2 124M: ragged pieces of tensors
        _case(name="gpt2_124m_shard8_adamw", shards=8, scale=65536.0),
        # GPT-2 124M mixed precision with loss scaling and clipping: the headline step
        _case(name="gpt2_124m_adamw", scale=65536.0),
        # GPT-2 774M: gradients beyond the Infinity Cache
        _case(name="gpt2_774m_adamw", scale=65536.0, **large),
        # GPT-2 1558M in full fp32: the largest step
        _case(name="gpt2_1558m_adamw_fp32", n_layer=48, d_model=1600, mode="fp32"),
        # SGD with momentum on a mixed store made for it
        _case(name="gpt2_124m_sgdm", opt="sgdm", layout="sgd", scale=65536.0),
        # the reference's own storage and optimizer: plain SGD on bf16 tensors
        _case(name="gpt2_774m_sgd_bf16", opt="sgd", mode="bf16", clip=0.0, **large),
        # a whole iteration behind a backward that hands over buckets, the norm from their sums
        _case(name="gpt2_124m_backward", kind="backward", scale=65536.0, sums=True),
        # gradient accumulation over four micro-batches in full precision
        _case(name="nanogpt_char_micro4_fp32", kind="backward", mode="fp32", source="fp32",
              micro=4, **nano),
        # master, m and v out to device tensors and another checkpoint's back in
        _case(name="gpt2_124m_transfer", kind="transfer"),
    ]


def draw(rng):
    """Another case of the same ranges: sizes from the MLP's to the largest listed model's."""
    kind = rng.choice(["step"] * 6 + ["backward"] * 3 + ["transfer"])
    c = _case(kind=kind)
    c["table"] = rng.choice(["gpt"] * 5 + ["ragged"] * 2 + ["mlp"])
    limit = MAX_PARAMS if kind == "step" else 300_000_000
    if c["table"] == "mlp":
        for key, lo, hi in (("d_in", 16, 4096), ("d_hidden", 64, 8192), ("d_out", 2, 4096)):
            c[key] = _log_int(rng, lo, hi)
    elif c["table"] == "ragged":
        c["n_tensors"] = _log_int(rng, 10, 1500)
        c["mean_numel"] = _log_int(rng, 300, 60_000)
    else:
        while True:
            c.update(n_layer=_log_int(rng, 2, 48), d_model=_log_int(rng, 60, 1700),
                     vocab=_log_int(rng, 65, 50257), ctx=_log_int(rng, 64, 2048))
            if sum(_table(c)[2]) <= limit:
                break
        if kind == "step" and rng.random() < 0.25:
            c["shards"] = rng.choice([2, 4, 8])
    c["mode"], c["layout"], c["opt"] = rng.choice(
        [("mixed", "default", "adamw")] * 4 + [("fp32", "default", "adamw")] * 3 +
        [("mixed", "sgd", "sgdm"), ("mixed", "default", "sgdm"), ("fp32", "default", "sgdm"),
         ("mixed", "sgd", "sgd"), ("fp32", "default", "sgd"), ("bf16", "default", "sgd")])
    c["clip"] = rng.choice([0.0, 1.0, 1.0, 1.0])
    c["scale"] = rng.choice([0.0, 1024.0, 65536.0]) if c["mode"] != "fp32" else 0.0
    if kind == "step":
        c["groups"] = 2 if rng.random() < 0.15 else 1
        c["captured"] = c["groups"] == 1 and rng.random() < 0.2
    elif kind == "backward":
        c["source"] = "fp32" if c["mode"] == "fp32" else rng.choice(["bf16", "bf16", "fp32"])
        c["micro"] = rng.choice([1, 1, 2, 4])
        c["sums"] = bool(c["clip"] or c["scale"]) and rng.random() < 0.6
    else:
        c.update(opt="adamw", layout="default", mode="fp32" if c["mode"] == "fp32" else "mixed")
    return c


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _table(c):
    """(shapes, decay flags, element counts) of a case's tensors."""
    if c["table"] == "mlp":
        i, h, o = c["d_in"], c["d_hidden"], c["d_out"]
        shapes = [(i, h), (h,), (h, o), (o,)]
    elif c["table"] == "ragged":
        # odd sizes spread over two orders of magnitude, matrices and vectors alike
        r = random.Random(1000 * c["n_tensors"] + c["mean_numel"])
        shapes = []
        for k in range(c["n_tensors"]):
            n = max(1, int(c["mean_numel"] * math.exp(r.uniform(-2.3, 1.2))))
            rows = r.choice([1, 3, 4, 7, 8])
            shapes.append((n,) if k % 3 == 2 else (rows, max(1, n // rows)))
    else:
        shapes = [s for _, s in configs.gpt2_params(c["n_layer"], c["d_model"], c["vocab"],
                                                    c["ctx"])]
        if c["shards"] > 1:
            return _last_shard(shapes, c["shards"])
    return shapes, [len(s) >= 2 for s in shapes], [math.prod(s) for s in shapes]


def _last_shard(shapes, shards):
    """The last of `shards` equal ranges of the flat store, as 1-D pieces of its tensors."""
    spans, at = [], 0
    for s in shapes:
        spans.append((at, math.prod(s), len(s) >= 2))
        at += -(-math.prod(s) // 64) * 64
    lo = (shards - 1) * (-(-(-(-at // shards)) // 64) * 64)
    pieces = [(o + n - max(o, lo), d) for o, n, d in spans if o + n > lo]
    return [(n,) for n, _ in pieces], [d for _, d in pieces], [n for n, _ in pieces]


def _offsets(numels):
    """Where each tensor starts in the flat store (64-element alignment), and the total."""
    at, out = 0, []
    for n in numels:
        out.append(at)
        at += -(-n // 64) * 64
    return out, at


def _inputs(c, seed):
    """Flat device arrays of the case's values, zeros in the padding: weights, Adam's moments,
    gradients (scaled, in the store's gradient type), another state for transfers, and the
    sources a backward hands over."""
    _, _, numels = _table(c)
    offsets, total = _offsets(numels)
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(std):
        x = torch.empty(total, dtype=torch.float32, device="cuda").normal_(0, std, generator=gen)
        for o, n, end in zip(offsets, numels, offsets[1:] + [total]):
            if o + n < end:
                x[o + n:end] = 0
        return x

    scale = c["scale"] or 1.0
    grad = torch.float32 if c["mode"] == "fp32" else torch.bfloat16
    v = {"p": randn(WEIGHT_STD)}
    if c["opt"] == "adamw":
        v["m"] = randn(0.3 * GRAD_STD)
        v["v"] = randn(GRAD_STD).square_()
    v["g"] = randn(GRAD_STD * scale).to(grad)
    if c["kind"] == "transfer":
        v["p2"], v["m2"], v["v2"] = randn(WEIGHT_STD), randn(GRAD_STD), randn(GRAD_STD).square_()
    elif c["kind"] == "backward":
        src = torch.bfloat16 if c["source"] == "bf16" else torch.float32
        v["src"] = [randn(GRAD_STD * scale / c["micro"]).to(src) for _ in range(c["micro"])]
    return v


def _view(store, which):
    """Device memory of one of the store's flat buffers, as its layout addresses it: weights and
    gradients flat, optimizer state by 64-element groups.  The tensor keeps the store, which owns
    the memory, alive."""
    base, group, stride = store.layout(which)
    flat = which in (ttperf.BUF_PARAM, ttperf.BUF_GRAD)
    two = flat and store.mode != ttperf._lib.MODE_FP32
    size = 2 if two else 4

    class _Device:
        __cuda_array_interface__ = {
            "data": (base, False), "typestr": "<u2" if two else "<f4", "version": 3,
            "shape": (store.total,) if flat else (store.total // group, group),
            "strides": (size,) if flat else (stride * size, size)}

    t = torch.as_tensor(_Device(), device=f"cuda:{store.device}")
    t = t.view(torch.bfloat16) if two else t
    t.owner = store
    return t


def _optimizers(c, store):
    """One optimizer over the store, or two over its alternating tensors."""
    clip = c["clip"] or None
    out = []
    for k in range(c["groups"]):
        params = store.parameters()[k::c["groups"]]
        lr = (LR if c["opt"] == "adamw" else SGD_LR) / (k + 1)
        if c["opt"] == "adamw":
            out.append(ttperf.AdamW(params, lr=lr, betas=BETAS, eps=EPS, weight_decay=WD,
                                    max_grad_norm=clip))
        elif c["opt"] == "sgdm":
            out.append(ttperf.SGD(params, lr=lr, momentum=MOMENTUM, weight_decay=WD,
                                  max_grad_norm=clip))
        else:
            out.append(ttperf.SGD(params, lr=lr, max_grad_norm=clip))
    return out


def _step(opts, **kw):
    """All optimizers' steps; the last one moves the loss scale."""
    for o in opts[:-1]:
        o.step(update_scale=False, **kw)
    opts[-1].step(**kw)


def prepare(case, seed):
    c = case
    gc.collect()  # an earlier store's memory goes back before this one is made
    shapes, decay, numels = _table(c)
    vals = _inputs(c, seed)
    store = ttperf.ParamStore(shapes, mode=c["mode"], decay=decay, layout=c["layout"])
    stream = torch.cuda.Stream() if c["captured"] else torch.cuda.current_stream()
    store.set_stream(stream)
    if c["scale"]:
        store.configure_scaler(True, init_scale=c["scale"])
    every = ttperf.ALL_TENSORS
    if c["mode"] == "bf16":
        store.upload(ttperf.BUF_PARAM, every, vals["p"].to(torch.bfloat16))
    else:
        store.upload(ttperf.BUF_MASTER, every, vals["p"])
    if c["opt"] == "adamw":
        store.upload(ttperf.BUF_EXP_AVG, every, vals["m"])
        store.upload(ttperf.BUF_EXP_AVG_SQ, every, vals["v"])
    if c["groups"] == 1:
        store.step_count = T0
    s = {"case": c, "store": store, "stream": stream}
    if c["kind"] == "transfer":
        s["state"] = [vals[k] for k in ("p2", "m2", "v2")]
        s["out"] = [torch.empty_like(x) for x in s["state"]]
        s["views"] = [_view(store, b) for b in (ttperf.BUF_PARAM, ttperf.BUF_MASTER,
                                                ttperf.BUF_EXP_AVG, ttperf.BUF_EXP_AVG_SQ)]
        return s
    # a training program that is under way: it has taken a step
    s["opts"] = opts = _optimizers(c, store)
    store.upload(ttperf.BUF_GRAD, every, vals["g"])
    _step(opts)
    bufs = {"param": ttperf.BUF_PARAM, "grad": ttperf.BUF_GRAD}
    if c["mode"] == "mixed":
        bufs["master"] = ttperf.BUF_MASTER
    if c["opt"] == "adamw":
        bufs.update(exp_avg=ttperf.BUF_EXP_AVG, exp_avg_sq=ttperf.BUF_EXP_AVG_SQ)
    elif c["opt"] == "sgdm":
        bufs["momentum"] = ttperf.BUF_MOMENTUM
    s["views"] = {k: _view(store, b) for k, b in bufs.items()}
    if c["kind"] == "backward":
        offsets, _ = _offsets(numels)
        s["micro"] = [[(idx, [src[offsets[i]:offsets[i] + numels[i]] for i in idx])
                       for idx in _buckets(numels, src.element_size())] for src in vals["src"]]
    elif c["captured"]:
        store.sync()
        store.begin_capture()
        _step(opts)
        s["graph"] = store.end_capture()
    return s


def _buckets(numels, esize):
    """Tensor indices in backward order (last first), about BUCKET_BYTES per bucket."""
    out, size = [[]], 0
    for i in reversed(range(len(numels))):
        if out[-1] and (size >= BUCKET_BYTES or len(out[-1]) == BUCKET_TENSORS):
            out.append([])
            size = 0
        out[-1].append(i)
        size += numels[i] * esize
    return out


def run(state):
    s = state
    c, store = s["case"], s["store"]
    if c["kind"] == "transfer":
        bufs = (ttperf.BUF_MASTER, ttperf.BUF_EXP_AVG, ttperf.BUF_EXP_AVG_SQ)
        for which, out in zip(bufs, s["out"]):
            store.download(which, out=out)
        for which, x in zip(bufs, s["state"]):
            store.upload(which, ttperf.ALL_TENSORS, x)
        return {"out": s["out"], "store": s["views"]}
    if c["kind"] == "backward":
        opt = s["opts"][0]
        opt.zero_grad()
        for k, micro in enumerate(s["micro"]):
            sums = c["sums"] and k == len(s["micro"]) - 1
            for idx, grads in micro:
                store.accumulate_grads(idx, grads, sums=sums)
        opt.step(tensor_sums=c["sums"])
    elif c["captured"]:
        s["graph"].replay()
    else:
        _step(s["opts"])
    return s["views"]


def work(case):
    c = case
    n = sum(_table(c)[2])
    g = 4 if c["mode"] == "fp32" else 2
    copy = 2 if c["mode"] == "mixed" else 0
    if c["kind"] == "transfer":
        return {"bytes": (2 * 12 + 2 * 12 + copy) * n, "flops": n}
    # fp32 state read and written, the bf16 copy written, the gradients read
    state = {"adamw": 3, "sgdm": 2, "sgd": 1}[c["opt"]]
    per = g + (2 * 2 if c["mode"] == "bf16" else state * 8 + copy)
    flops = {"adamw": 18, "sgdm": 8, "sgd": 3}[c["opt"]]
    if c["kind"] == "backward":
        # the sources read, the gradients written once (and used from there)
        per += c["micro"] * (2 if c["source"] == "bf16" else 4)
        flops += c["micro"]
    return {"bytes": per * n, "flops": flops * n}


def tolerance(case):
    if case["kind"] == "transfer":
        return "exact"  # copies, and the bf16 rounding of the weights
    if case["mode"] == "fp32":
        # measured against exact(): at most 8e-8 on any output
        return {"rel": 4e-7, "max": 1e-5}
    # fp32 values as above; where they move by an ulp, a bf16 weight may round to its other
    # neighbour (2^-8 away), at a few in 10^5 places: 4e-3 * sqrt(5e-5)
    return {"rel": 1e-4, "max": 1e-2}


def exact(case, seed):
    """run()'s outputs of a new state in 64 bits (the step before it included)."""
    c = case
    _, decay, numels = _table(c)
    offsets, total = _offsets(numels)
    vals = _inputs(c, seed)
    if c["kind"] == "transfer":
        first = [vals[k].double() for k in ("p", "m", "v")]
        second = [vals[k].double() for k in ("p2", "m2", "v2")]
        return {"out": first, "store": [second[0]] + [x.view(-1, 64) for x in second]}
    p = (vals["p"].to(torch.bfloat16) if c["mode"] == "bf16" else vals["p"]).double()
    adam, mom = c["opt"] == "adamw", c["opt"] == "sgdm"
    m = vals["m"].double() if adam else torch.zeros_like(p) if mom else None
    v = vals["v"].double() if adam else None
    lr0 = LR if adam else SGD_LR
    if c["mode"] == "bf16":  # the reference's lr fill of the bf16 gradient's type
        lr0 = float(torch.tensor(lr0).to(torch.bfloat16))
    for it in range(2):
        if it == 1 and c["kind"] == "backward":
            g = sum(x.double() for x in vals["src"])
        else:
            g = vals["g"].double()
        grad = g
        g = g / (c["scale"] or 1.0)
        for k in range(c["groups"]):
            mine = range(len(numels))[k::c["groups"]]
            norm = math.sqrt(sum(g[offsets[i]:offsets[i] + numels[i]].square().sum().item()
                                 for i in mine)) if c["clip"] else 0.0
            coef = min(1.0, c["clip"] / (norm + 1e-6)) if c["clip"] else 1.0
            t = (T0 if c["groups"] == 1 else 0) + it + 1
            lr = lr0 / (k + 1)  # (a power of two: exact after the bf16 rounding too)
            for i in mine:
                a = slice(offsets[i], offsets[i] + numels[i])
                pi, gi = p[a], g[a] * coef
                if adam:
                    if decay[i]:
                        pi.mul_(1 - lr * WD)
                    m[a].mul_(BETAS[0]).add_(gi, alpha=1 - BETAS[0])
                    v[a].mul_(BETAS[1]).addcmul_(gi, gi, value=1 - BETAS[1])
                    den = (v[a] / (1 - BETAS[1] ** t)).sqrt_().add_(EPS)
                    pi.addcdiv_(m[a], den, value=-lr / (1 - BETAS[0] ** t))
                elif mom:
                    if decay[i]:
                        gi = gi + WD * pi
                    m[a].copy_(gi if it == 0 else MOMENTUM * m[a] + gi)
                    pi.sub_(m[a], alpha=lr)
                else:
                    pi.sub_(gi, alpha=lr)
    out = {"param": p, "grad": grad}
    if c["mode"] == "mixed":
        out["master"] = p.view(-1, 64)
    if adam:
        out.update(exp_avg=m.view(-1, 64), exp_avg_sq=v.view(-1, 64))
    elif mom:
        out["momentum"] = m.view(-1, 64)
    return out
