"""The work this library does for its users, as cases to time and to compare.

Two kinds of call make up a training or inference program on this library:

* ``kind="linear"``: one Monarch projection through ``butterfly_blk``, the call a patched ``MonarchLinear``
  makes -- the forward alone (generation, evaluation, prompt processing) or forward and backward (training).
* ``kind="step"``: one optimizer step over a model's Monarch factors and its embedding / norm / head tensors,
  ``MonarchMuonOptimizer`` or ``CoatStateMonarchMuon`` (FP8 states), with or without ``clip_grad_norm_`` before it.

Sizes are those of the benchmark configurations (toy, 257M, 1.3B, 6.89B: ``monarch_muon_amd/workloads.py``) and of a
124M model (width 768).  A step over a large model takes a few of its equal layers, which is one rank's share of a
step sharded by block ownership, and the same share of the AdamW elements.
"""
import math

import torch

from monarch_muon_amd import CoatStateMonarchMuon, MonarchMuonOptimizer, QuantizationConfig, butterfly_blk
from monarch_muon_amd.workloads import factor_shapes

DEV = "cuda"
LR, MU, BETAS, WD, EPS = 0.02, 0.95, (0.9, 0.95), 0.1, 1e-8
NS_A, NS_B, NS_C, NS_STEPS = 3.4445, -4.7750, 2.0315, 5
ADAM_STEP = 10          # steps the AdamW moments have seen before the pass
CLIP = 1.0
PAD = 256               # elements: tensors start where separate allocations would


def _linear(name, tokens, din, dout, nb, train):
    return dict(name=name, kind="linear", tokens=tokens, din=din, dout=dout, nb=nb, train=train)


def _step(name, width, hidden, nb, layers, adamw, param, mom, ns, clip):
    """``param`` / ``mom``: "bf16", "f32" (``mom`` also "fp8"); ``ns``: "bf16" or "own" (Newton-Schulz in the momentum
    dtype); ``adamw``: elements of the embedding and head tensors."""
    return dict(name=name, kind="step", width=width, hidden=hidden, nb=nb, layers=layers, adamw=adamw, param=param,
                mom=mom, ns=ns, clip=clip)


def listed():
    return [
        # generation: a batch of eight sequences, one token each, through the 6.89B gate / up projection
        _linear("decode-6.89b-up", 8, 4096, 11008, 4, False),
        # prompt processing / evaluation: a ragged batch of prompts through the 6.89B down projection
        _linear("prefill-6.89b-down", 3001, 11008, 4096, 4, False),
        # training the toy model: one short ragged micro-batch, where launches and host time count
        _linear("train-toy-up", 1000, 512, 1376, 2, True),
        # training the 257M model: its down projection on 16 sequences of 1024
        _linear("train-257m-down", 16384, 2736, 1024, 2, True),
        # training the 1.3B model: an attention projection at the benchmark's micro-batch (4 x 1024)
        _linear("train-1.3b-q", 4096, 2048, 2048, 4, True),
        # training the 6.89B model: the gate / up projection at the same micro-batch
        _linear("train-6.89b-up", 4096, 4096, 11008, 4, True),
        # the toy configuration whole: fp32 everywhere, Newton-Schulz in fp32, gradients clipped as the trainer does
        _step("step-toy-f32", 512, 1376, 2, 2, 2 * 50304 * 512, "f32", "f32", "own", True),
        # a 124M model (width 768, two blocks of 384): block sides that are no multiple of a 256-wide tile
        _step("step-124m-bf16", 768, 2048, 2, 12, 2 * 50304 * 768, "bf16", "f32", "bf16", True),
        # the 257M configuration whole: bf16 parameters, fp32 momentum, clipped
        _step("step-257m-bf16", 1024, 2736, 2, 24, 2 * 50304 * 1024, "bf16", "f32", "bf16", True),
        # a sixth of the 1.3B model in fp32 (the pretraining copy of the optimizer)
        _step("step-1.3b-f32", 2048, 5504, 4, 4, 2 * 50304 * 2048 // 6, "f32", "f32", "own", False),
        # a sixteenth of the 6.89B model with FP8 optimizer states
        _step("step-6.89b-fp8", 4096, 11008, 4, 2, 2 * 50304 * 4096 // 16, "bf16", "fp8", "bf16", False),
        # an eighth of the 6.89B model, the headline configuration: one rank's share of an 8-way sharded step
        _step("step-6.89b-bf16", 4096, 11008, 4, 4, 2 * 50304 * 4096 // 8, "bf16", "f32", "bf16", False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.5:
        nb = rng.choice([2, 4, 4])
        unit = 32 * nb                                   # the layers' short block side is a multiple of it
        q = unit * rng.randint(-(-192 // unit), 1024 // unit)
        other = 8 * rng.randint(q // 8, 22 * q // 64)    # long block side: up to 2.75 times the short one
        din, dout = rng.choice([(q, q), (q, other), (other, q)])
        train = rng.random() < 0.6
        most = 8192 * 1024 // q if train else 16384
        tokens = _log(rng, 64 if train else 1, most)
        return _unnamed(_linear("", tokens, nb * din, nb * dout, nb, train))
    nb = rng.choice([2, 4])
    block = 8 * rng.randint(12, 128)                     # 96 .. 1024
    other = 8 * rng.randint(block // 8, 22 * block // 64)
    kind = rng.choice(["bf16", "bf16", "bf16mom", "f32", "fp8"])
    param, mom, ns = {"bf16": ("bf16", "f32", "bf16"), "bf16mom": ("bf16", "bf16", "bf16"),
                      "f32": ("f32", "f32", "own"), "fp8": ("bf16", "fp8", "bf16")}[kind]
    c = _step("", nb * block, nb * other, nb, 1, 0, param, mom, ns, rng.random() < 0.5)
    # layers: spread up to the largest listed step's work (fp32 products run on a slower unit)
    limit = (9e11 if kind == "f32" else 5e12) / _step_flops(c)
    c["layers"] = max(1, min(24, _log(rng, 1, max(1.01, limit))))
    c["adamw"] = _log(rng, 100_000, 40_000_000)
    return _unnamed(c)


def _unnamed(c):
    return {k: v for k, v in c.items() if k != "name"}


# ---------------------------------------------------------------------------
# linear
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _linear_inputs(c, seed):
    g = _gen(seed)
    s1, s2 = factor_shapes(c["din"], c["dout"], c["nb"])
    x = torch.randn(c["tokens"], s1[0] * s1[2], generator=g, device=DEV).bfloat16()
    w1 = (torch.randn(s1, generator=g, device=DEV) / s1[2] ** 0.5).bfloat16()
    w2 = (torch.randn(s2, generator=g, device=DEV) / s2[2] ** 0.5).bfloat16()
    dy = torch.randn(c["tokens"], s2[0] * s2[1], generator=g, device=DEV).bfloat16() if c["train"] else None
    return x, w1, w2, dy


def _linear_exact(c, seed):
    x, w1, w2, dy = (t.double() if t is not None else None for t in _linear_inputs(c, seed))
    nb, q, p = w1.shape
    s, B = w2.shape[1], x.shape[0]

    def mm(a, b):
        return torch.stack([u @ v for u, v in zip(a, b)])

    xb = x.view(B, nb, p).transpose(0, 1)                         # (k, B, p)
    out1 = mm(xb, w1.transpose(1, 2)).transpose(0, 1).reshape(B, nb * q)
    t = out1.view(B, q, nb).permute(2, 0, 1)                      # feature i nb + l of a row: block l, entry i
    y = mm(t, w2.transpose(1, 2)).permute(1, 2, 0).reshape(B, s * nb)
    if dy is None:
        return [y]
    d = dy.view(B, s, nb).permute(2, 0, 1)                        # (l, B, s)
    dw2 = mm(d.transpose(1, 2), t)
    dt = mm(d, w2)                                                # (l, B, q)
    d1 = dt.permute(1, 2, 0).reshape(B, nb, q).transpose(0, 1)    # (k, B, q)
    dx = mm(d1, w1).transpose(0, 1).reshape(B, nb * p)
    return [y, dx, mm(d1.transpose(1, 2), xb), dw2]


# ---------------------------------------------------------------------------
# step
# ---------------------------------------------------------------------------
_DT = {"bf16": torch.bfloat16, "f32": torch.float32}


def _muon_shapes(c):
    w, h, nb = c["width"], c["hidden"], c["nb"]
    layer = [s for din, dout in ((w, w),) * 4 + ((w, h), (w, h), (h, w)) for s in factor_shapes(din, dout, nb)]
    return layer * c["layers"]


def _adamw_shapes(c):
    half = c["adamw"] // 2
    return [(half,)] + [(c["width"],)] * (2 * c["layers"] + 1) + [(c["adamw"] - half,)]


def _slots(shapes):
    """(offsets, total) of tensors laid one after the other, each at a multiple of PAD elements."""
    at, offs = 0, []
    for s in shapes:
        offs.append(at)
        at += -(-math.prod(s) // PAD) * PAD
    return offs, at


def _views(flat, shapes, offs):
    return [flat[o:o + math.prod(s)].view(s) for s, o in zip(shapes, offs)]


class _Space:
    """Parameters, gradients and states of one update type: one storage each, the tensors views of it."""

    def __init__(self, c, shapes, seed):
        self.shapes = shapes
        self.offs, self.n = _slots(shapes)
        pd, g = _DT[c["param"]], _gen(seed)
        live = torch.zeros(self.n, dtype=torch.bool, device=DEV)
        for s, o in zip(shapes, self.offs):
            live[o:o + math.prod(s)] = True

        def rand(scale, dtype):
            return torch.where(live, torch.randn(self.n, generator=g, device=DEV) * scale, 0.0).to(dtype)

        self.live = live
        self.p = rand(0.02, pd)
        self.g = rand(1e-3, pd)
        self.rand = rand

    def fp8(self, value):
        """FP8 codes and metadata of ``value`` (groups of 128): code * scale, the codec's expand 1 form."""
        v = value.view(-1, 128)
        scale = (v.abs().amax(1) / 448.0).clamp_min(1e-30)
        codes = (v / scale[:, None]).to(torch.float8_e4m3fn).view(-1)
        return [codes, scale, torch.ones_like(scale), torch.ones_like(scale)]


def _spaces(c, seed):
    muon = _Space(c, _muon_shapes(c), seed)
    adam = _Space(c, _adamw_shapes(c), seed + 7919)
    if c["mom"] == "fp8":
        muon.buf = muon.fp8(muon.rand(1e-3, torch.float32))
        adam.m = adam.fp8(adam.rand(1e-3, torch.float32))
        adam.v = adam.fp8(adam.rand(1e-3, torch.float32).square())
    else:
        muon.buf = muon.rand(1e-3, _DT[c["mom"]])
        adam.m = adam.rand(1e-3, adam.p.dtype)
        adam.v = adam.rand(1e-3, torch.float32).square().to(adam.p.dtype)
    return muon, adam


_META = ("", "scale_", "expand_", "sqrt_minmax_")


def _put(state, name, store, shape, off):
    if torch.is_tensor(store):
        state[name] = store[off:off + math.prod(shape)].view(shape)
        return
    n = math.prod(shape)
    state[name] = store[0][off:off + n].view(shape)
    for key, t in zip(_META[1:], store[1:]):
        state[key + name] = t[off // 128:off // 128 + -(-n // 128)]


def _step_prepare(c, seed):
    muon, adam = _spaces(c, seed)
    params = []
    for sp in (muon, adam):
        ps = []
        for p, g in zip(_views(sp.p, sp.shapes, sp.offs), _views(sp.g, sp.shapes, sp.offs)):
            p = p.detach().requires_grad_(True)
            p.grad = g
            ps.append(p)
        params.append(ps)
    kw = dict(lr=LR, momentum=MU, adamw_betas=BETAS, adamw_weight_decay=WD, adamw_eps=EPS,
              ns_dtype=torch.bfloat16 if c["ns"] == "bf16" else None)
    if c["mom"] == "fp8":
        opt = CoatStateMonarchMuon(*params, qargs=QuantizationConfig(), **kw)
    else:
        opt = MonarchMuonOptimizer(*params, **kw)
    for p, s, o in zip(params[0], muon.shapes, muon.offs):
        _put(opt.state[p], "momentum_buffer", muon.buf, s, o)
    for p, s, o in zip(params[1], adam.shapes, adam.offs):
        st = opt.state[p]
        st["step"] = ADAM_STEP
        _put(st, "exp_avg", adam.m, s, o)
        _put(st, "exp_avg_sq", adam.v, s, o)
    return dict(opt=opt, clip=c["clip"], outputs=dict(p=muon.p, buf=muon.buf, adam_p=adam.p, m=adam.m, v=adam.v))


def _ns_exact(x):
    """Newton-Schulz of a stack of equal blocks (N, r, c), as the quintic states it."""
    x = x / (x.norm(dim=(1, 2), keepdim=True) + 1e-7)
    tall = x.shape[1] > x.shape[2]
    if tall:
        x = x.transpose(1, 2).contiguous()
    for _ in range(NS_STEPS):
        a = torch.bmm(x, x.transpose(1, 2).contiguous())
        x = NS_A * x + torch.bmm(NS_B * a + NS_C * torch.bmm(a, a), x)
    return x.transpose(1, 2) if tall else x


def _step_exact(c, seed):
    muon, adam = _spaces(c, seed)
    gm, ga = muon.g.double(), adam.g.double()
    out = {}
    if c["clip"]:
        total = torch.sqrt(gm.square().sum() + ga.square().sum())
        coef = torch.clamp(CLIP / (total + 1e-6), max=1.0)
        gm, ga = gm * coef, ga * coef
        out["norm"] = total

    def dq(store):
        if torch.is_tensor(store):
            return store.double()
        return (store[0].float().view(-1, 128) * store[1][:, None]).double().view(-1)

    buf = dq(muon.buf) * MU + gm
    p = muon.p.double()
    by_shape = {}
    for s, o in zip(muon.shapes, muon.offs):
        by_shape.setdefault(s, []).append(o)
    for s, offs in by_shape.items():
        n = math.prod(s)
        for o in offs:
            u = _ns_exact(buf[o:o + n].view(s))
            p[o:o + n] -= (LR * math.sqrt(s[1] / s[2])) * u.reshape(-1)
    m = dq(adam.m) * BETAS[0] + (1 - BETAS[0]) * ga
    v = dq(adam.v) * BETAS[1] + (1 - BETAS[1]) * ga * ga
    t = ADAM_STEP + 1
    ap = adam.p.double() * (1 - LR * WD)
    ap = ap - LR / (1 - BETAS[0] ** t) * m / (v.sqrt() / math.sqrt(1 - BETAS[1] ** t) + EPS)
    ap = torch.where(adam.live, ap, 0.0)
    fp8 = c["mom"] == "fp8"
    out.update(p=p, buf=None if fp8 else buf, adam_p=ap, m=None if fp8 else m, v=None if fp8 else v)
    return out


def _step_flops(c):
    """Newton-Schulz of every block: symmetric products counted once, in the cheaper of the chain and its form on
    m x m matrices."""
    total = 0.0
    for s in _muon_shapes(c):
        m, n = min(s[1], s[2]), max(s[1], s[2])
        chain = NS_STEPS * (m * m * n + m ** 3 + 2 * m * m * n)
        gram = 6 * m * m * n + 14 * m ** 3
        total += s[0] * float(min(chain, gram))
    return total


# ---------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "step":
        return _step_prepare(case, seed)
    x, w1, w2, dy = _linear_inputs(case, seed)
    if case["train"]:
        for t in (x, w1, w2):
            t.requires_grad_(True)
    return dict(x=x, w1=w1, w2=w2, dy=dy)


def run(state):
    if "opt" in state:
        opt, out = state["opt"], dict(state["outputs"])
        if state["clip"]:
            out["norm"] = opt.clip_grad_norm_(CLIP)
        opt.step()
        return out
    x, w1, w2, dy = state["x"], state["w1"], state["w2"], state["dy"]
    if dy is None:
        with torch.no_grad():
            return [butterfly_blk(x, w1, w2)]
    y = butterfly_blk(x, w1, w2)
    return [y.detach(), *torch.autograd.grad(y, (x, w1, w2), dy)]


def exact(case, seed):
    return _step_exact(case, seed) if case["kind"] == "step" else _linear_exact(case, seed)


def work(case):
    if case["kind"] == "linear":
        (nb, q, p), (_, s, _) = factor_shapes(case["din"], case["dout"], case["nb"])
        tok, w = case["tokens"], nb * (q * p + s * q)
        io = 2.0 * (tok * nb * (p + s) + w)
        flops = 2.0 * tok * w
        # training: dy read too, dx and the weight gradients written; two more products per factor
        return dict(bytes=2 * io, flops=3 * flops) if case["train"] else dict(bytes=io, flops=flops)
    size = {"bf16": 2.0, "f32": 4.0, "fp8": 1.0 + 12 / 128}
    pd, md = size[case["param"]], size[case["mom"]]
    ad = md if case["mom"] == "fp8" else pd
    nm = sum(math.prod(s) for s in _muon_shapes(case))
    na = sum(math.prod(s) for s in _adamw_shapes(case))
    # each read once: parameter, gradient, states; each written once: parameter, states
    return dict(bytes=nm * (3 * pd + 2 * md) + na * (3 * pd + 4 * ad), flops=_step_flops(case))


def tolerance(case):
    # four times the distance measured from the 64-bit values: bf16 projections 2.3e-3, bf16 steps up to 2.4e-3
    # (4.6e-3 where the clipping coefficient is rounded to bf16); fp32 steps 1.1e-7 with 32-bit sums over up to
    # 1376 terms and five iterations behind them
    if case["kind"] == "linear":
        return {"rel": 8e-3, "max": 0.05}
    if case["param"] == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["mom"] == "fp8":       # a value on a rounding tie takes the next code: an eighth of its size
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.1}
