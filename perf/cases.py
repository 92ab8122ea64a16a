"""Timed cases of the optimizer step: the calls a training loop makes, over the range of models it makes them for.

Every case goes through the package's public classes (``step()``, ``assign_hooks`` +
backward + ``reassign_grad_buffer``, ``SRLinear`` forward and backward, ``newton_schulz``).
A case's parameters are views of one flat buffer, as in a program that keeps flat
parameters, so that outputs stay few however many tensors a model has.

    listed()                the cases that are always measured
    draw(rng)               one more case of the same ranges
    prepare(case, seed)     what a program has before the call, on the GPU
    run(state)              one pass; its outputs
    work(case)              bytes and flops that the pass cannot do without
    tolerance(case)         how far another correct implementation may be
    exact(case, seed)       the outputs in 64 bits, in plain torch
"""
import math
import random

import torch

import muon_sr_amd as M

DEV = "cuda"
NS_A, NS_B, NS_C = 3.4445, -4.7750, 2.0315


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the 8-bit step of one flat parameter of 2^28 elements: an embedding of 131072 x 2048
        dict(name="adamw8bit_flat_268M", kind="adamw8bit", tensors=1, numel=1 << 28, block=256, noise="philox8"),
        # a whole model on the 8-bit optimizer: 8-bit matrices, bf16 moments for the embedding and
        # the norm vectors, one call per tensor
        dict(name="adamw8bit_8L_d2048", kind="adamw8bit", layers=8, d=2048, ffn=5632, kv=2048, vocab=32000,
             block=256, noise="philox8"),
        # odd sizes, a smaller quantization block and the reference's noise stream
        dict(name="adamw8bit_odd_block64", kind="adamw8bit", tensors=6, numel=30000001, block=64, noise="triton"),
        # bf16-moment AdamW over a small GPT (8 layers, d 384, vocab 16384): latency and launches
        dict(name="adamw_8L_d384", kind="adamw", layers=8, d=384, ffn=1536, kv=384, vocab=16384, centralization=0.0,
             noise="philox8"),
        # bf16-moment AdamW with gradient centralization on one large embedding
        dict(name="adamw_central_128256x4096", kind="adamw", tensors=1, rows=128256, cols=4096, centralization=1.0,
             noise="philox8"),
        # Muon with stacked momenta: 16 layers of a d = 2048 transformer
        dict(name="muon_16L_d2048", kind="muon", layers=16, d=2048, ffn=5632, kv=2048, batch_ns=True,
             noise="philox8"),
        # Muon with its default options (one parameter after the other): 2 layers of the same
        dict(name="muon_each_2L_d2048", kind="muon", layers=2, d=2048, ffn=5632, kv=2048, batch_ns=False,
             noise="philox8"),
        # the smallest hybrid step: 4 matrices of 256 x 256, two vectors and a 512 x 256 embedding
        dict(name="hybrid_4x256", kind="hybrid", tensors=4, rows=256, cols=256, vocab=512, bits=16, batch_ns=True,
             noise="philox8"),
        # the hybrid step at Llama-3-8B's shapes, 4 of its 32 layers, 8-bit AdamW for the
        # embedding and the head
        dict(name="hybrid_4L_llama3_8b", kind="hybrid", layers=4, d=4096, ffn=14336, kv=1024, vocab=128256, bits=8,
             batch_ns=True, noise="philox8"),
        # two micro-batches accumulated by the backward hooks, at the same model's layer shapes
        dict(name="accum_4L_llama3_8b", kind="accum", layers=4, d=4096, ffn=14336, kv=1024, micro=2,
             noise="philox8"),
        # a linear layer's forward and backward with the fused accumulation, two micro-batches
        dict(name="srlinear_2048x2048_t4096", kind="srlinear", fin=2048, fout=2048, tokens=4096, micro=2,
             noise="philox8"),
        # Newton-Schulz alone on the 8 MLP matrices of the small GPT
        dict(name="ns_8x1536x384", kind="ns", batch=8, rows=1536, cols=384),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """Log-uniform in [lo, hi]: half of them multiples of `step`, the others as they come."""
    v = _log(rng, lo, hi)
    return max(step, v // step * step) if rng.random() < 0.5 else v


def draw(rng):
    noise = "philox8" if rng.random() < 0.75 else "triton"
    kind = rng.choice(["adamw8bit", "adamw", "muon", "muon", "hybrid", "accum", "srlinear", "ns"])
    if kind == "adamw8bit":
        return dict(kind=kind, tensors=rng.randint(1, 10), numel=_size(rng, 5000, 1 << 25, 256),
                    block=rng.choice([64, 128, 256, 256, 256, 512, 2048]), noise=noise)
    if kind == "adamw":
        return dict(kind=kind, tensors=rng.randint(1, 10), rows=_size(rng, 16, 8192, 64), cols=_size(rng, 16, 4096, 64),
                    centralization=rng.choice([0.0, 0.0, 1.0]), noise=noise)
    if kind == "muon" or kind == "ns":
        while True:
            rows, cols, n = _size(rng, 48, 6144, 128), _size(rng, 48, 6144, 128), rng.randint(1, 12)
            if n * _ns_flops(rows, cols) < 8e12:
                break
        if kind == "ns":
            return dict(kind=kind, batch=n, rows=rows, cols=cols)
        return dict(kind=kind, tensors=n, rows=rows, cols=cols, batch_ns=rng.random() < 0.5, noise=noise)
    if kind == "hybrid":
        d = _size(rng, 128, 2048, 64)
        return dict(kind=kind, layers=rng.randint(1, 6), d=d, ffn=_size(rng, d, 4 * d, 64), kv=d // rng.choice([1, 4]),
                    vocab=_size(rng, 500, 50000, 64), bits=rng.choice([8, 16]), batch_ns=rng.random() < 0.5,
                    noise=noise)
    if kind == "accum":
        return dict(kind=kind, tensors=rng.randint(1, 24), rows=_size(rng, 16, 8192, 64), cols=_size(rng, 16, 4096, 64),
                    micro=rng.randint(1, 4), noise=noise)
    return dict(kind=kind, fin=256 * _log(rng, 1, 24), fout=256 * _log(rng, 1, 24), tokens=128 * _log(rng, 2, 64),
                micro=rng.randint(1, 2), noise=noise)


# ---------------------------------------------------------------------------
# shapes and inputs
# ---------------------------------------------------------------------------

def _matrices(case):
    """The weight matrices (for Muon: its parameters)."""
    if "layers" in case:
        d, f, k = case["d"], case["ffn"], case["kv"]
        return [(d, d), (k, d), (k, d), (d, d), (f, d), (f, d), (d, f)] * case["layers"]
    if "rows" in case:
        return [(case["rows"], case["cols"])] * case["tensors"]
    return [(case["numel"] // (i + 1) + i,) for i in range(case["tensors"])]


def _others(case):
    """Embedding (and head) first, then the norm vectors."""
    v = case.get("vocab", 0)
    if "layers" in case:
        d = case["d"]
        emb = [(v, d)] * (2 if case.get("bits") == 8 else 1) if v else []
        return emb + [(d,)] * (2 * case["layers"])
    return [(v, case["cols"]), (case["cols"],), (case["cols"],)] if v else []


def _numel(shape):
    return math.prod(shape)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(shape, std, gen):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16).mul_(std)


def _flat(shapes, fill):
    """One flat buffer and its views, each 128-byte aligned, filled with fill(shape)."""
    at, offs = 0, []
    for s in shapes:
        offs.append(at)
        at += -(-_numel(s) // 64) * 64
    flat = torch.zeros(at, dtype=torch.bfloat16, device=DEV)
    views = [flat[o:o + _numel(s)].view(s) for o, s in zip(offs, shapes)]
    for v, s in zip(views, shapes):
        v.copy_(fill(s))
    return flat, views


def _params(shapes, gen):
    flat, views = _flat(shapes, lambda s: _randn(s, 0.02, gen))
    ps = [torch.nn.Parameter(v) for v in views]
    return flat, ps


def _grads(ps, std, gen):
    for p in ps:
        p.grad = _randn(p.shape, std, gen)


def _flatten_states(opt, ps, keys):
    """Moves the optimizer's state tensors of `keys` into one flat buffer per (key, dtype)."""
    out = {}
    for key in keys:
        for dt in (torch.bfloat16, torch.uint8, torch.float32):
            own = [p for p in ps if opt.state[p].get(key) is not None and opt.state[p][key].dtype == dt]
            if not own:
                continue
            at, offs = 0, []
            for p in own:
                offs.append(at)
                at += -(-opt.state[p][key].numel() // 64) * 64
            flat = torch.zeros(at, dtype=dt, device=DEV)
            for p, o in zip(own, offs):
                t = opt.state[p][key]
                v = flat[o:o + t.numel()].view(t.shape)
                v.copy_(t)
                opt.state[p][key] = v
            out["%s_%s" % (key, str(dt).split(".")[1])] = flat
    return out


def _stacks(opt, ps):
    """The stacked momenta of a batch_ns optimizer, one per shape."""
    out = {}
    for p in ps:
        out.setdefault("momentum_%dx%d" % tuple(p.shape), opt.state[p]["momentum_buffer"]._base)
    return out


def _adam_shapes(case):
    return _matrices(case) + _others(case)


MUON = dict(lr=0.02, momentum=0.95, weight_decay=0.01)
ADAM = dict(lr=3e-4, betas=(0.9, 0.95), eps=1e-10, weight_decay=0.1)
ADAM8 = dict(lr=3e-4, betas=(0.9, 0.95), eps=1e-10, weight_decay=0.01)
WARM = 2   # steps taken before the timed one, so that moments and block scales are those of a run


class _Emit(torch.autograd.Function):
    """A backward pass that delivers the given gradients to the parameters (as fresh
    tensors, so autograd hands them on without a copy)."""

    @staticmethod
    def forward(ctx, grads, out, *params):
        ctx.grads = grads
        return out.view_as(out)

    @staticmethod
    def backward(ctx, g):
        return (None, None, *[t.view_as(t) for t in ctx.grads])


def prepare(case, seed):
    gen = _gen(seed)
    random.seed(seed)   # the accumulator draws its seeds from `random`
    kind = case["kind"]
    M.set_sr_noise(case.get("noise", "philox8"))
    st = dict(case=case)
    if kind == "ns":
        st["G"] = _randn((case["batch"], case["rows"], case["cols"]), 1e-3, gen)
        return st
    if kind == "srlinear":
        lin = M.SRLinear(case["fin"], case["fout"], bias=False, device=DEV, dtype=torch.bfloat16)
        with torch.no_grad():
            lin.weight.copy_(_randn((case["fout"], case["fin"]), 0.02, gen))
        st["lin"] = lin
        st["x"] = [_randn((case["tokens"], case["fin"]), 1.0, gen).requires_grad_() for _ in range(case["micro"])]
        st["dy"] = [_randn((case["tokens"], case["fout"]), 1e-3, gen) for _ in range(case["micro"])]
        return st
    if kind == "accum":
        _, ps = _params(_matrices(case) + _others(case), gen)
        model = torch.nn.ParameterList(ps)
        M.TritonSRAccumulator.assign_hooks(model)
        st["model"], st["ps"] = model, ps
        st["grads"] = [[_randn(p.shape, 1e-4, gen) for p in ps] for _ in range(case["micro"])]
        st["one"] = torch.ones((), device=DEV)
        return st
    if kind == "muon":
        st["flat"], ps = _params(_matrices(case), gen)
        opt = M.TritonMuonSR(ps, batch_ns=case["batch_ns"], **MUON)
        muon, adam = ps, []
    elif kind == "hybrid":
        muon_shapes, adam_shapes = _matrices(case), _others(case)
        st["flat"], ps = _params(muon_shapes + adam_shapes, gen)
        muon, adam = ps[:len(muon_shapes)], ps[len(muon_shapes):]
        extra = dict(optim_bits=8) if case["bits"] == 8 else {}
        opt = M.TritonMuonSRWithAuxAdam([dict(params=muon, use_muon=True, **MUON),
                                         dict(params=adam, use_muon=False, **ADAM, **extra)],
                                        batch_ns=case["batch_ns"])
    elif kind == "adamw":
        st["flat"], ps = _params(_adam_shapes(case), gen)
        opt = M.TritonAdamW(ps, centralization=case["centralization"], **ADAM)
        muon, adam = [], ps
    else:
        shapes = _adam_shapes(case)
        st["flat"], ps = _params(shapes, gen)
        n8 = len(_matrices(case))
        groups = [dict(params=ps[:n8], optim_bits=8)] + ([dict(params=ps[n8:], optim_bits=16)] if ps[n8:] else [])
        opt = M.TritonAdamW8bit(groups, block_size=case["block"], **ADAM8)
        muon, adam = [], ps
    for _ in range(WARM):
        _grads(ps, 1e-3, gen)
        opt.step()
    st["states"] = {}
    if muon and case["batch_ns"]:
        st["states"].update(_stacks(opt, muon))
    elif muon:
        st["states"].update(_flatten_states(opt, muon, ["momentum_buffer"]))
    st["states"].update(_flatten_states(opt, adam, ["ema", "ema_squared", "state1", "state2", "absmax1", "absmax2"]))
    _grads(ps, 1e-3, gen)
    st["opt"], st["ps"], st["muon"], st["adam"] = opt, ps, muon, adam
    return st


def run(st):
    case = st["case"]
    M.set_sr_noise(case.get("noise", "philox8"))
    kind = case["kind"]
    if kind == "ns":
        return M.newton_schulz(st["G"], 5)
    if kind == "srlinear":
        lin = st["lin"]
        lin.weight.grad = None
        ys, dxs = [], []
        for x, dy in zip(st["x"], st["dy"]):
            x.grad = None
            y = lin(x)
            y.backward(dy)
            ys.append(y.detach())
            dxs.append(x.grad)
        M.TritonSRAccumulator.reassign_grad_buffer(lin)
        return dict(y=ys, dx=dxs, dw=lin.weight.grad)
    if kind == "accum":
        for p in st["ps"]:
            p.grad = None
        for grads in st["grads"]:
            _Emit.apply(grads, st["one"], *st["ps"]).backward()
        M.TritonSRAccumulator.reassign_grad_buffer(st["model"])
        return [p.grad for p in st["ps"]]
    st["opt"].step()
    return dict(params=st["flat"], **st["states"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------

def _ns_flops(rows, cols):
    """Five iterations: A = X X^T (symmetric: half of 2 m^2 n), A A (symmetric: half of 2 m^3), B X (2 m^2 n)."""
    m, n = min(rows, cols), max(rows, cols)
    return 5.0 * (3 * m * m * n + m * m * m)


def work(case):
    kind = case["kind"]
    if kind == "ns":
        return dict(bytes=4.0 * case["batch"] * case["rows"] * case["cols"],
                    flops=case["batch"] * _ns_flops(case["rows"], case["cols"]))
    if kind == "srlinear":
        i, o, t, k = case["fin"], case["fout"], case["tokens"], case["micro"]
        # forward, input gradient, weight gradient; x, dy, W in, y, dx and the accumulator out
        return dict(bytes=2.0 * (k * (2 * t * i + 2 * t * o) + 2 * i * o + (2 * k - 1) * i * o), flops=6.0 * k * t * i * o)
    if kind == "accum":
        n = sum(_numel(s) for s in _matrices(case) + _others(case))
        return dict(bytes=float(n) * (6 * case["micro"] - 2), flops=0.0)
    nm = 0
    flops = 0.0
    if kind in ("muon", "hybrid"):
        nm = sum(_numel(s) for s in _matrices(case))
        flops = sum(_ns_flops(*s) for s in _matrices(case))
    by = 10.0 * nm                                    # p and momentum read and written, gradient read
    if kind == "hybrid":
        for s in _others(case):
            n = _numel(s)
            by += n * 10.0625 if case["bits"] == 8 and n >= 4096 else n * 14.0
    elif kind == "adamw":
        by += 14.0 * sum(_numel(s) for s in _adam_shapes(case))
    elif kind == "adamw8bit":
        by += sum(_numel(s) * (10.0 + 16.0 / case["block"] if _numel(s) >= 4096 else 14.0) for s in _matrices(case))
        by += 14.0 * sum(_numel(s) for s in _others(case))
    return dict(bytes=by, flops=flops)


def tolerance(case):
    kind = case["kind"]
    # Element-wise steps: every fp32 operation is rounded as IEEE says and the noise is a
    # function of (seed, offset), so another correct implementation gives the same bits.
    if kind in ("adamw", "adamw8bit", "accum"):
        return "exact"
    # bf16 Newton-Schulz with its sums in another order (the same matrix with its columns
    # permuted: 0.3e-2 to 0.5e-2).
    if kind == "ns":
        return dict(rel=1.5e-2, max=0.2)
    # one bf16 rounding of 32-bit sums whose order is free
    if kind == "srlinear":
        return dict(rel=4e-3, max=0.2)
    # Muon: the update's 0.5e-2 reaches the parameters as one-ulp flips of the stochastic
    # rounding where it moves a value past its noise threshold; momenta and the AdamW
    # states of the hybrid are the same bits.
    return dict(rel=2e-3, max=0.2)


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------

def _ns64(U):
    X = U.double()
    tall = X.shape[-2] > X.shape[-1]
    X = X.transpose(-2, -1).contiguous() if tall else X
    X = X / (X.norm(dim=(-2, -1), keepdim=True) + 1e-7)
    for _ in range(5):
        A = X @ X.transpose(-2, -1).contiguous()
        B = NS_B * A + NS_C * (A @ A)
        X = NS_A * X + B @ X
    return X.transpose(-2, -1).contiguous() if tall else X


def _adam64(p, g, m, v, step, lr, b1, b2, eps, wd):
    """m, v, and the two forms of the parameter: decay before the update, or after it."""
    m = b1 * m + (1 - b1) * g
    v = b2 * v + (1 - b2) * g * g
    upd = lr / (1 - b1 ** step) * m / (v.sqrt() / (1 - b2 ** step) ** 0.5 + eps)
    return m, v, p * (1 - lr * wd) - upd, (p - lr / (1 - b1 ** step) * m / (v.sqrt() / (1 - b2 ** step) ** 0.5 + eps)) * (1 - lr * wd)


def _dequant(codes, qmap, absmax, block):
    n = codes.numel()
    return qmap.double()[codes.reshape(-1).long()] * absmax.double().repeat_interleave(block)[:n]


def _block_max(x, block):
    x = x.abs().reshape(-1)
    pad = -x.numel() % block
    return torch.cat([x, x.new_zeros(pad)]).view(-1, block).amax(1)


def _put(flat, view, value):
    """Writes `value` at the place that `view` has in its flat buffer's 64-bit twin."""
    flat[view.storage_offset():view.storage_offset() + view.numel()] = value.reshape(-1).to(flat.dtype)


def exact(case, seed):
    kind = case["kind"]
    w = work(case)
    if w["flops"] > 1.5e13 or w["bytes"] > 1.2e10:
        return None
    st = prepare(case, seed)
    if kind == "ns":
        return _ns64(st["G"])
    if kind == "srlinear":
        W = st["lin"].weight.detach().double()
        y = [x.detach().double() @ W.t().contiguous() for x in st["x"]]
        dx = [dy.double() @ W for dy in st["dy"]]
        dw = sum(dy.double().t().contiguous() @ x.detach().double() for x, dy in zip(st["x"], st["dy"]))
        return dict(y=y, dx=dx, dw=dw)
    if kind == "accum":
        return [sum(g[i].double() for g in st["grads"]) for i in range(len(st["ps"]))]
    opt = st["opt"]
    out = dict(params=torch.zeros_like(st["flat"], dtype=torch.float64))
    for key, t in st["states"].items():
        out[key] = torch.zeros(t.shape, dtype=torch.float64, device=DEV) if t.is_floating_point() else None
    for p in st["muon"]:
        g, b = p.grad.double(), opt.state[p]["momentum_buffer"]
        nb = b.double() + (1 - MUON["momentum"]) * (g - b.double())
        u = g + MUON["momentum"] * (nb - g)
        scale = max(1.0, p.shape[0] / p.shape[1]) ** 0.5
        new = p.detach().double() * (1 - MUON["lr"] * MUON["weight_decay"]) - MUON["lr"] * scale * _ns64(u)
        _put(out["params"], p, new)
        key = "momentum_%dx%d" % tuple(p.shape) if case["batch_ns"] else "momentum_buffer_bfloat16"
        _put(out[key].view(-1), b, nb)
    for p in st["adam"]:
        s = opt.state[p]
        hyper = ADAM8 if kind == "adamw8bit" else ADAM
        (b1, b2), args = hyper["betas"], (s["step"] + 1, hyper["lr"], *hyper["betas"], hyper["eps"], hyper["weight_decay"])
        g, q = p.grad.double(), p.detach().double()
        if "ema" in s:
            if case.get("centralization"):
                g = g - g.mean(dim=tuple(range(1, g.dim())), keepdim=True) * case["centralization"]
            m, v, new, _ = _adam64(q, g, s["ema"].double(), s["ema_squared"].double(), *args)
            _put(out["ema_bfloat16"], s["ema"], m)
            _put(out["ema_squared_bfloat16"], s["ema_squared"], v)
        elif s["optim_bits"] == 16:
            m, v, _, new = _adam64(q, g, s["state1"].double(), s["state2"].double(), *args)
            _put(out["state1_bfloat16"], s["state1"], m)
            _put(out["state2_bfloat16"], s["state2"], v)
        else:
            bs = s["block_size"]
            m0 = _dequant(s["state1"], s["qmap1"], s["absmax1"], bs).view(p.shape)
            v0 = _dequant(s["state2"], s["qmap2"], s["absmax2"], bs).view(p.shape)
            m, v, _, new = _adam64(q, g, m0, v0, *args)
            _put(out["absmax1_float32"], s["absmax1"], _block_max(m, bs))
            _put(out["absmax2_float32"], s["absmax2"], _block_max(v, bs))
        _put(out["params"], p, new)
    return out
