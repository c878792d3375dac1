"""Performance cases of Video Sparse Attention on one GPU.

Each case is one call that a video model makes of this package: the whole op on
block-ordered tokens (``mi355x_vsa``), the fine branch on a route of the
caller's own (``mi355x_sparse_attention``) or the op on raster-order tokens
(``mi355x_vsa_tiled``), as inference or as a training step that returns the
gradients too.

A case's keys:

* ``op``: "full", "route" or "raster"; ``train``; ``dtype``; ``B``, ``H``, ``D``;
* ``block``: the block's shape "TxHxW"; ``qb``, ``kb``: query and key blocks
  (block-ordered ops), or ``latent``: the raster grid "TxHxW";
* ``topk``; ``gate``: "none", "token" ([B, H, S, 1]) or "full" ([B, H, S, D]);
* ``ragged``: 0 for full blocks, n for every n-th block (and the last) three
  quarters full, as the edge tiles of a grid are;
* ``layout``: "head" for [B, H, S, D] memory, "token" for per-head views of
  [B, S, H, D] memory (a projection's output);
* ``skew``: exponent of the Zipf popularity of key blocks in a caller's route.
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "simple-vsa_amd"))

import vsa_mi355x  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEFAULTS = dict(op="full", train=True, dtype="bf16", B=1, H=1, D=128, block="4x4x4", qb=0, kb=0,
                latent="", topk=1, gate="none", ragged=0, layout="head", skew=0.0)


def _case(name=None, **kw):
    c = dict(DEFAULTS, **kw)
    if c["latent"]:
        grid, tile = _triple(c["latent"]), _triple(c["block"])
        c["qb"] = c["kb"] = math.prod(math.ceil(g / t) for g, t in zip(grid, tile))
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # a short clip or a low-resolution preview at inference, where a call's own cost counts
        _case("infer_short", train=False, H=8, D=64, qb=32, kb=32, topk=4),
        # the same at a unit test's size, in 32 bits, as a training step: the smallest call
        _case("train_tiny_fp32", dtype="fp32", H=2, D=64, qb=16, kb=16, topk=2),
        # a short training clip straight from the projections, with the gate
        _case("train_short", H=12, qb=64, kb=64, topk=8, gate="full", layout="token"),
        # the small benchmark shape: a 12-head model, the last block partly filled
        _case("train_small", H=12, block="1x1x256", qb=64, kb=64, topk=8, gate="token",
              ragged=64),
        # the headline benchmark: a 40-head video model's training step at 41k tokens
        _case("train_video", H=40, block="4x8x8", qb=160, kb=160, topk=20, gate="full"),
        # serving the longest videos: 92k tokens, the forward alone, partly filled edge blocks
        _case("infer_long", train=False, H=40, block="1x1x256", qb=360, kb=360, topk=45,
              ragged=8),
        # a caller's own route that favours some key blocks, small blocks and heads
        _case("train_routes_skewed", op="route", H=24, D=64, block="1x1x64", qb=640, kb=640,
              topk=32, skew=1.2),
        # raster-order tokens of a 12-head model: a grid whose edge tiles are partly empty
        _case("train_raster", op="raster", H=12, latent="21x30x52", topk=78, gate="full",
              layout="token"),
        # wide heads
        _case("train_wide_head", H=8, D=256, block="4x8x8", qb=64, kb=64, topk=8),
        # a run in 32 bits, as one checks a model's training against
        _case("train_fp32", dtype="fp32", H=12, block="1x1x256", qb=64, kb=64, topk=8,
              gate="token", ragged=64),
        # few queries against a longer context, in half precision, on a caller's route
        _case("train_cross_fp16", op="route", dtype="fp16", H=16, block="2x8x8", qb=40, kb=96,
              topk=12, ragged=12),
        # a tile volume and head dim that no kernel is made for
        _case("train_odd", H=10, D=80, block="3x3x3", qb=300, kb=300, topk=38, gate="full",
              ragged=10),
    ]


def _triple(text):
    return tuple(int(x) for x in text.split("x"))


def _be(case):
    return math.prod(_triple(case["block"]))


def _flops(case):
    """Two products per selected pair of tokens in the forward, five more backward."""
    be = _be(case)
    fwd = 4.0 * case["B"] * case["H"] * case["qb"] * case["topk"] * be * be * case["D"]
    return fwd * (3.5 if case["train"] else 1.0)


def _cost(case):
    """Seconds that a pass would take at rates that this card reaches easily: what
    keeps a drawn case below the largest listed one."""
    be, d = _be(case), case["D"]
    kbe, kd = (next(x for x in (64, 128, 256) if v <= x) for v in (be, d))
    pad = (kbe / be) ** 2 * kd / d
    rate = 6e13 if case["dtype"] == "fp32" else {64: 4e14, 128: 5e14, 256: 6e14}[kbe]
    return _flops(case) * pad / rate


def draw(rng):
    while True:
        op = rng.choice(["full", "full", "full", "route", "raster"])
        train = rng.random() < 0.65
        dtype = rng.choice(["bf16"] * 6 + ["fp16", "fp32"])
        block = rng.choice(["4x4x4", "4x4x4", "2x8x8", "4x8x8", "4x8x8", "3x3x3", "4x4x5", "2x5x7"])
        d = rng.choice([64, 128, 128, 128, 256, 72, 96, 160])
        h = rng.choice([2, 3, 5, 8, 12, 16, 24, 40])
        b = rng.choice([1, 1, 1, 2])
        be = math.prod(_triple(block))
        kw = dict(op=op, train=train, dtype=dtype, block=block, D=d, H=h, B=b,
                  gate="none" if op == "route" else rng.choice(["none", "token", "full"]))
        if op == "raster":
            n = int(math.exp(rng.uniform(math.log(1000), math.log(60000))))
            t = rng.randint(3, 33)
            w = max(4, int(math.sqrt(n / t * 1.7)))
            kw["latent"] = "%dx%dx%d" % (t, max(3, n // (t * w)), w)
            kw["layout"] = rng.choice(["head", "token"])
        else:
            n = int(math.exp(rng.uniform(math.log(1000), math.log(92160))))
            kw["kb"] = max(3, n // be)
            kw["qb"] = max(2, kw["kb"] // rng.choice([2, 3])) if rng.random() < 0.2 else kw["kb"]
            kw["ragged"] = rng.choice([0, 0, 3, 8, kw["kb"]])
            if op == "full" and kw["qb"] == kw["kb"]:
                kw["layout"] = rng.choice(["head", "token"])
            if op == "route":
                kw["skew"] = rng.choice([0.0, 0.7, 1.2])
        case = _case(**kw)
        if not 3 <= case["kb"] <= 2000:
            continue
        case["topk"] = max(1, min(case["kb"], int(case["kb"] * rng.choice([0.0625, 0.125, 0.125, 0.25]))))
        if _cost(case) <= 1.2e-2:
            return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _sizes(n, be, ragged, device):
    vbs = torch.full((n,), be, dtype=torch.int32, device=device)
    if ragged:
        vbs[ragged - 1::ragged] = max(1, be * 3 // 4)
        vbs[-1] = max(1, be * 3 // 4)
    return vbs


def _slots(case, device):
    """Raster token of each padded tile slot (-1: padding), and the tiles' sizes."""
    (T, H, W), (a, b, c) = _triple(case["latent"]), _triple(case["block"])
    n = [math.ceil(x / y) for x, y in zip((T, H, W), (a, b, c))]
    t, h, w = (torch.arange(m * y, device=device).view(m, y) for m, y in zip(n, (a, b, c)))
    t = t.view(n[0], 1, 1, a, 1, 1)
    h = h.view(1, n[1], 1, 1, b, 1)
    w = w.view(1, 1, n[2], 1, 1, c)
    inside = ((t < T) & (h < H) & (w < W)).reshape(-1, a * b * c)
    token = ((t * H + h) * W + w).expand(*n, a, b, c).reshape(-1, a * b * c)
    # a tile's tokens come first, its padding after them
    order = torch.argsort((~inside).to(torch.int8), dim=1, stable=True)
    token = torch.where(inside, token, -1).gather(1, order)
    return token.reshape(-1), inside.sum(1).to(torch.int32)


def _inputs(case, seed):
    """q, k, v, gate, dout (head-major), the block sizes and the route.  Tokens are
    unit noise around their block's own value, as neighbouring tokens of a video
    are alike; padding tokens are zero, as tile() leaves them."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    B, H, D, be = case["B"], case["H"], case["D"], _be(case)
    dt = DTYPES[case["dtype"]]

    def rand(*shape):
        return torch.randn(shape, generator=g, device=dev)

    if case["op"] == "raster":
        slots, _ = _slots(case, dev)
        s_out = math.prod(_triple(case["latent"]))
        block_of = torch.empty(s_out, dtype=torch.long, device=dev)
        real = slots >= 0
        block_of[slots[real]] = torch.arange(slots.numel(), device=dev)[real] // be
        qvbs = vbs = None
    else:
        vbs = _sizes(case["kb"], be, case["ragged"], dev)
        qvbs = _sizes(case["qb"], be, case["ragged"], dev)

    def tokens(nb, sizes, width, offset=0.5):
        if sizes is None:
            x = rand(B, H, block_of.numel(), width)
            return (x + offset * rand(B, H, nb, width)[:, :, block_of]).to(dt)
        x = rand(B, H, nb, be, width)
        x += offset * rand(B, H, nb, 1, width)
        x *= (torch.arange(be, device=dev) < sizes[:, None])[..., None]
        return x.view(B, H, nb * be, width).to(dt)

    q, k, v = (tokens(n, s, D) for n, s in ((case["qb"], qvbs), (case["kb"], vbs),
                                            (case["kb"], vbs)))
    dout = tokens(case["qb"], qvbs, D, 0.0) if case["train"] else None
    gate = None
    if case["gate"] != "none":
        shape = (B, H, q.shape[2], D if case["gate"] == "full" else 1)
        gate = torch.rand(shape, generator=g, device=dev).to(dt)
    sel = None
    if case["op"] == "route":
        # topk key blocks a row without repeats, block i as likely as 1 / rank(i)^skew
        perm = torch.argsort(torch.rand(case["kb"], generator=g, device=dev))
        logp = -case["skew"] * torch.log1p(perm.double())
        u = torch.rand((B, H, case["qb"], case["kb"]), generator=g, device=dev,
                       dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
        sel = torch.topk(logp - torch.log(-torch.log(u)), case["topk"], dim=-1).indices.int()
    return q, k, v, gate, dout, vbs, qvbs, sel


def prepare(case, seed):
    q, k, v, gate, dout, vbs, qvbs, sel = _inputs(case, seed)
    if case["layout"] == "token":
        raster = case["op"] == "raster"   # takes [B, S, H, D] itself; the others a view of it
        q, k, v, gate, dout = (None if x is None else x.transpose(1, 2).contiguous()
                               if raster else x.transpose(1, 2).contiguous().transpose(1, 2)
                               for x in (q, k, v, gate, dout))
    leaves = [x for x in (q, k, v, gate) if x is not None]
    if case["train"]:
        for x in leaves:
            x.requires_grad_()
    return dict(case=case, q=q, k=k, v=v, gate=gate, dout=dout, vbs=vbs, qvbs=qvbs, sel=sel,
                leaves=leaves, block=_triple(case["block"]))


def _forward(s):
    c = s["case"]
    if c["op"] == "route":
        return vsa_mi355x.mi355x_sparse_attention(s["q"], s["k"], s["v"], s["sel"], s["vbs"],
                                                  block_size=s["block"])
    if c["op"] == "raster":
        return vsa_mi355x.mi355x_vsa_tiled(s["q"], s["k"], s["v"], _triple(c["latent"]),
                                           c["topk"], tile_size=s["block"],
                                           compress_attn_weight=s["gate"],
                                           token_major=c["layout"] == "token")
    return vsa_mi355x.mi355x_vsa(s["q"], s["k"], s["v"], s["vbs"], s["qvbs"], c["topk"],
                                 block_size=s["block"], compress_attn_weight=s["gate"])


def run(state):
    if not state["case"]["train"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    return [out.detach(), *torch.autograd.grad(out, state["leaves"], state["dout"])]


def work(case):
    e = DTYPES[case["dtype"]].itemsize
    B, H, D, be = case["B"], case["H"], case["D"], _be(case)
    if case["latent"]:
        sq = skv = math.prod(_triple(case["latent"]))
    else:
        sq, skv = case["qb"] * be, case["kb"] * be
    g = {"none": 0, "token": 1, "full": D}[case["gate"]]
    read = sq * D + 2 * skv * D + sq * g
    moved = read + sq * D                           # the inputs and out
    if case["train"]:
        moved += read + sq * D                      # dout and the gradients
    return {"bytes": B * H * e * moved, "flops": _flops(case)}


def tolerance(case):
    # four times the error of out and of the gradients against 64 bits
    return {"rel": {"bf16": 1e-2, "fp16": 1.5e-3, "fp32": 1e-5}[case["dtype"]]}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

def _mm(a, b):
    return torch.matmul(a, b.contiguous())


def _t(x):
    return x.transpose(-2, -1).contiguous()


def _mean(x, sizes, be):
    nb = x.shape[0] // be
    on = (torch.arange(be, device=x.device) < sizes[:, None])[..., None]
    return (x.view(nb, be, -1) * on).sum(1) / sizes.clamp(min=1)[:, None], on


def _route(qc, kc, topk, scale, dt):
    """Top-K of the coarse scores as the op's contract rounds them: block means and
    both roundings of the scores in the input type, ties to the smaller block."""
    s = (_mm(qc.to(dt).double(), _t(kc.to(dt).double())).to(dt).float() * scale).to(dt)
    return torch.sort(s.double(), dim=-1, descending=True, stable=True).indices[:, :topk]


def _fine(q, k, v, sel, vbs, be, scale, dout=None):
    """One head's fine branch on the routed blocks, and its gradients."""
    nb, tk = sel.shape
    d = q.shape[1]
    kbl, vbl = k.view(-1, be, d), v.view(-1, be, d)
    ok = torch.arange(be, device=q.device) < vbs[:, None]
    out, dq = torch.empty_like(q), torch.empty_like(q)
    dk, dv = torch.zeros_like(kbl), torch.zeros_like(vbl)
    step = max(1, (1 << 27) // (be * tk * be))
    for i in range(0, nb, step):
        s = sel[i:i + step].long()
        n = s.shape[0]
        rows = slice(i * be, (i + n) * be)
        qs, ks, vs = q[rows].view(n, be, d), kbl[s].view(n, tk * be, d), vbl[s].view(n, tk * be, d)
        p = _mm(qs, _t(ks)) * scale
        p.masked_fill_(~ok[s].view(n, 1, tk * be), -math.inf)
        p = torch.softmax(p, dim=-1)
        o = _mm(p, vs)
        out[rows] = o.view(-1, d)
        if dout is None:
            continue
        g = dout[rows].view(n, be, d)
        dv.index_add_(0, s.reshape(-1), _mm(_t(p), g).view(-1, be, d))
        ds = _mm(g, _t(vs))
        ds -= (o * g).sum(-1, keepdim=True)
        ds *= p
        ds *= scale
        dq[rows] = _mm(ds, ks).view(-1, d)
        dk.index_add_(0, s.reshape(-1), _mm(_t(ds), qs).view(-1, be, d))
    return out, dq, dk.view_as(k), dv.view_as(v)


def _head(case, q, k, v, gate, dout, vbs, qvbs, sel, dt):
    be, scale = _be(case), 1.0 / math.sqrt(case["D"])
    if case["op"] == "route":
        out, dq, dk, dv = _fine(q, k, v, sel, vbs, be, scale, dout)
        return out, dq, dk, dv, None
    (qc, qon), (kc, kon), (vc, _) = _mean(q, qvbs, be), _mean(k, vbs, be), _mean(v, vbs, be)
    sel = _route(qc, kc, case["topk"], scale, dt)
    out, dq, dk, dv = _fine(q, k, v, sel, vbs, be, scale, dout)
    p = torch.softmax(_mm(qc, _t(kc)) * scale, dim=-1)
    oc = _mm(p, vc)
    wide = oc.repeat_interleave(be, 0)
    out += wide if gate is None else wide * gate
    if dout is None:
        return out, None, None, None, None
    dgate = None
    if gate is not None:
        dgate = dout * wide
        dgate = dgate.sum(-1, keepdim=True) if gate.shape[-1] == 1 else dgate
    doc = (dout if gate is None else dout * gate).view(-1, be, dout.shape[-1]).sum(1)
    dp = _mm(doc, _t(vc))
    ds = p * (dp - (dp * p).sum(-1, keepdim=True)) * scale

    def spread(x, on, sizes):
        return ((x / sizes.clamp(min=1)[:, None])[:, None] * on).reshape(-1, x.shape[-1])

    dq += spread(_mm(ds, kc), qon, qvbs)
    dk += spread(_mm(_t(ds), qc), kon, vbs)
    dv += spread(_mm(_t(p), doc), kon, vbs)
    return out, dq, dk, dv, dgate


def exact(case, seed):
    q, k, v, gate, dout, vbs, qvbs, sel = _inputs(case, seed)
    dt, (B, H) = q.dtype, q.shape[:2]
    slots = None
    if case["op"] == "raster":
        slots, vbs = _slots(case, q.device)
        qvbs = vbs
        real = slots >= 0
        tile = slots.clamp(min=0)

    def at(x, b, h):
        if x is None:
            return None
        x = x[b, h].double()
        return x if slots is None else x[tile] * real[:, None]

    def back(x):
        if slots is None:
            return x
        y = x.new_empty((math.prod(_triple(case["latent"])), x.shape[-1]))
        y[slots[real]] = x[real]
        return y

    parts = []
    for b in range(B):
        for h in range(H):
            got = _head(case, *(at(x, b, h) for x in (q, k, v, gate, dout)), vbs, qvbs,
                        None if sel is None else sel[b, h], dt)
            parts.append([None if x is None else back(x) for x in got])
    outs = []
    for group in zip(*parts):
        if group[0] is None:
            continue
        x = torch.stack(group).view(B, H, *group[0].shape)
        if slots is not None and case["layout"] == "token":
            x = x.transpose(1, 2)
        outs.append(x)
    return outs if case["train"] else outs[0]
