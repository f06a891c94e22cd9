"""What the framework's performance is measured on: calls of its public entry
points as a user's program makes them, over the range of sizes, data types and
options that neighborhood-attention models use.

A case is a dict of plain values.  Extents, kernel sizes, dilations and
strides of several axes are texts such as ``"56x56"``; ``causal`` holds one
digit per axis.  ``op`` names the entry point:

* ``fused``  -- ``na1d`` / ``na2d`` / ``na3d`` (``grad``: with the backward);
* ``varlen`` -- ``na1d_varlen_gqa``: padded batch, grouped heads, global tokens;
* ``split``  -- ``na2d_qk`` -> softmax -> ``na2d_av``, the path of a layer with
  dropout on its attention weights;
* ``rpb``    -- ``extras.allin1``: QK with relative position bias -> softmax -> AV;
* ``layer``  -- ``nn.NeighborhoodAttention2D``, projections included.
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "natten-mlx_amd"))

import natten_amd  # noqa: E402
from natten_amd.extras import allin1  # noqa: E402

DEVICE = "cuda:0"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
FUSED = {1: natten_amd.na1d, 2: natten_amd.na2d, 3: natten_amd.na3d}


def _fused(name, dtype, batch, spatial, heads, dim, kernel, dilation="", stride="", causal="",
           kv_heads=0, grad=True, lse=False):
    rank = len(spatial.split("x"))
    ones = "x".join("1" * rank)
    return {"name": name, "op": "fused", "dtype": dtype, "batch": batch, "spatial": spatial,
            "heads": heads, "kv_heads": kv_heads or heads, "dim": dim, "kernel": kernel,
            "dilation": dilation or ones, "stride": stride or ones, "causal": causal or "0" * rank,
            "grad": grad, "lse": lse}


def _varlen(name, dtype, batch, length, heads, kv_heads, dim, kernel, dilation, extra):
    return {"name": name, "op": "varlen", "dtype": dtype, "batch": batch, "spatial": str(length),
            "heads": heads, "kv_heads": kv_heads, "dim": dim, "kernel": str(kernel),
            "dilation": str(dilation), "extra": extra}


def _split(name, dtype, batch, spatial, heads, dim, kernel, dilation):
    return {"name": name, "op": "split", "dtype": dtype, "batch": batch, "spatial": spatial,
            "heads": heads, "kv_heads": heads, "dim": dim, "kernel": kernel,
            "dilation": dilation}


def _rpb(name, batch, spatial, heads, dim, kernel, dilation):
    return {"name": name, "op": "rpb", "dtype": "f32", "batch": batch, "spatial": spatial,
            "heads": heads, "kv_heads": heads, "dim": dim, "kernel": kernel,
            "dilation": dilation}


def _layer(name, dtype, batch, spatial, heads, dim, kernel, dilation):
    return {"name": name, "op": "layer", "dtype": dtype, "batch": batch, "spatial": spatial,
            "heads": heads, "kv_heads": heads, "dim": dim, "kernel": kernel,
            "dilation": dilation}


def listed():
    return [
        # the quick start: one short sequence, where the call itself is the cost
        _fused("na1d quick start f32 fwd", "f32", 2, "64", 4, 32, "7", grad=False),
        # a training step of an image model's first stage
        _fused("na2d train bf16", "bf16", 4, "56x56", 4, 32, "7x7"),
        # the same in single precision, torch's default type, on an image
        # whose sides are no multiple of any tile
        _fused("na2d train f32 ragged", "f32", 2, "61x45", 8, 32, "7x7"),
        # a training step of a video model, causal in time, LSE kept
        _fused("na3d train bf16 causal", "bf16", 1, "16x32x32", 8, 64, "3x7x7", causal="100",
               lse=True),
        # long sequences of different lengths, grouped heads, global tokens
        _varlen("na1d varlen gqa f16", "f16", 8, 4096, 16, 4, 64, 63, 2, 16),
        # a pooling step: every second query, odd sides
        _fused("na2d strided train bf16", "bf16", 4, "57x75", 4, 64, "7x7", stride="2x2"),
        # a layer with dropout on its attention weights takes the split path
        _split("na2d split train bf16", "bf16", 4, "56x56", 4, 32, "7x7", "1x1"),
        # relative position bias, one and two axes (single precision only)
        _rpb("rpb 1d train f32", 8, "2048", 12, 12, "7", "2"),
        _rpb("rpb 2d train f32", 4, "56x56", 2, 32, "7x7", "1x1"),
        # a whole layer with its projections
        _layer("layer 2d train bf16", "bf16", 8, "56x56", 8, 32, "7x7", "2x2"),
        # a large image at inference, wide window
        _fused("na2d inference f16 large", "f16", 1, "384x384", 8, 64, "13x13", grad=False),
        # a window as long as the sequence: plain attention
        _fused("na1d dense train bf16", "bf16", 4, "4096", 16, 64, "4096"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _window(rng, kernels, extents, dilations):
    """Odd kernel sizes and dilations that fit their extents."""
    ks, ds = [], []
    k0, d0 = rng.choice(kernels), rng.choice(dilations)
    for e in extents:
        k, d = k0, d0
        while d > 1 and k * d > e:
            d -= 1
        while k > e:
            k -= 2
        ks.append(k)
        ds.append(d)
    return _text(ks), _text(ds)


def _text(values):
    return "x".join(str(v) for v in values)


def _draw(rng):
    kind = rng.randrange(11)
    half = rng.choice(("bf16", "bf16", "f16"))
    if kind == 0:  # inference, small to large, every type
        n = _log(rng, 64, 65536)
        dtype = rng.choice(("f32", "bf16", "f16"))
        if rng.random() < 0.5:
            ext = [n]
            k, d = _window(rng, (3, 7, 13, 31, 63), ext, (1, 2, 4))
        else:
            a = max(14, int(math.sqrt(n) * rng.uniform(0.7, 1.4)))
            ext = [a, max(14, n // a)]
            k, d = _window(rng, (3, 5, 7, 9, 13), ext, (1, 2, 4))
        return _fused("", dtype, rng.randint(1, 4), _text(ext), rng.choice((4, 8, 16)),
                      rng.choice((32, 64)), k, d, causal=rng.choice("001") + "0" * (len(ext) - 1),
                      grad=False)
    if kind == 1:  # training, images, 16 bits
        ext = [_log(rng, 14, 128), _log(rng, 14, 128)]
        k, d = _window(rng, (3, 5, 7, 7, 9, 13), ext, (1, 1, 2, 4))
        heads = rng.choice((2, 4, 8, 16))
        return _fused("", half, rng.randint(1, 8), _text(ext), heads, rng.choice((32, 64, 128)),
                      k, d, kv_heads=rng.choice((heads, heads, heads // 2)))
    if kind == 2:  # training, images, single precision
        ext = [_log(rng, 14, 96), _log(rng, 14, 96)]
        k, d = _window(rng, (3, 5, 7, 7, 9, 13), ext, (1, 1, 2, 4))
        return _fused("", "f32", rng.randint(1, 4), _text(ext), rng.choice((2, 4, 8)),
                      rng.choice((32, 32, 64)), k, d, causal=rng.choice(("00", "00", "10")))
    if kind == 3:  # training, video
        ext = [_log(rng, 6, 24), _log(rng, 14, 40), _log(rng, 14, 40)]
        k, d = _window(rng, (3, 5, 7), ext[1:], (1, 1, 2))
        return _fused("", rng.choice((half, half, "f32")), 1, _text(ext), rng.choice((4, 8)),
                      rng.choice((32, 64)), "3x" + k, "1x" + d, lse=rng.random() < 0.5,
                      causal=rng.choice(("100", "000")))
    if kind == 4:  # sequences of different lengths
        length, group = _log(rng, 512, 6000), rng.choice((1, 2, 4))
        kv = rng.choice((2, 4))
        return _varlen("", half, rng.randint(2, 8), length, kv * group, kv,
                       rng.choice((32, 64, 128)), rng.choice((7, 15, 31, 63)), rng.choice((1, 2)),
                       rng.choice((4, 16, 32)))
    if kind == 5:  # strided queries
        ext = [_log(rng, 16, 112), _log(rng, 16, 112)]
        k, _ = _window(rng, (3, 5, 7, 9), ext, (1,))
        s = rng.choice((2, 2, 3)) if "3" not in k.split("x") else 2
        return _fused("", rng.choice((half, half, "f32")), rng.randint(1, 6), _text(ext),
                      rng.choice((2, 4, 8)), rng.choice((32, 64)), k, stride=f"{s}x{s}")
    if kind == 6:
        ext = [_log(rng, 14, 80), _log(rng, 14, 80)]
        k, d = _window(rng, (3, 5, 7, 7), ext, (1, 1, 2, 4))
        return _split("", rng.choice((half, half, "f32")), rng.randint(1, 6), _text(ext),
                      rng.choice((2, 4, 8)), rng.choice((32, 32, 64)), k, d)
    if kind == 7:
        length = _log(rng, 200, 6000)
        k, d = _window(rng, (3, 5, 7), [length], (1, 2, 4, 8))
        return _rpb("", rng.randint(1, 12), str(length), rng.choice((4, 6, 12)),
                    rng.choice((8, 12, 16)), k, d)
    if kind == 8:
        ext = [_log(rng, 14, 80), _log(rng, 14, 80)]
        k, d = rng.choice((3, 5, 7, 7)), rng.choice((1, 1, 2))
        return _rpb("", rng.randint(1, 6), _text(ext), rng.choice((2, 4, 8)),
                    rng.choice((16, 32)), f"{k}x{k}", f"{d}x{d}")
    if kind == 9:
        ext = [_log(rng, 14, 72), _log(rng, 14, 72)]
        k, d = _window(rng, (3, 5, 7, 7), ext, (1, 1, 2, 4))
        return _layer("", rng.choice((half, half, "f32")), rng.randint(1, 8), _text(ext),
                      rng.choice((2, 4, 8, 16)), 32, k, d)
    n = _log(rng, 200, 5000)  # plain attention
    return _fused("", half, rng.randint(1, 4), str(n), rng.choice((4, 8, 16)),
                  rng.choice((32, 64, 128)), str(n))


def draw(rng):
    most = _cost(listed()[-1])
    while True:
        case = _draw(rng)
        case.pop("name")
        if _cost(case) <= most:
            return case


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


# ---------------------------------------------------------------------------

def _axes(case):
    """Per axis (extent, kernel, dilation, stride, causal)."""
    ext = [int(v) for v in case["spatial"].split("x")]
    ker = [int(v) for v in case["kernel"].split("x")]
    dil = [int(v) for v in case["dilation"].split("x")]
    st = [int(v) for v in case["stride"].split("x")] if "stride" in case else [1] * len(ext)
    ca = [c == "1" for c in case["causal"]] if "causal" in case else [False] * len(ext)
    return list(zip(ext, ker, dil, st, ca))


def _lengths(case):
    """The samples' lengths: spread evenly from a quarter of the padded one."""
    n, (length, k, d, _, _) = case["batch"], _axes(case)[0]
    lo = max(length // 4, k * d)
    return [lo + (length - lo) * (2 * i + 1) // (2 * n) for i in range(n)]


def _pairs(case):
    """Query-key pairs of one head over the batch."""
    axes = _axes(case)
    if case["op"] == "varlen":
        return sum(_lengths(case)) * (axes[0][1] + case["extra"])
    n = case["batch"]
    for ext, k, d, s, ca in axes:
        n *= sum(min(k, p // d + 1) if ca else k for p in range(0, ext, s))
    return n


def work(case):
    axes = _axes(case)
    size = 4 if case["dtype"] == "f32" else 2
    tok = case["batch"] * math.prod(a[0] for a in axes)
    otok = case["batch"] * math.prod(-(-a[0] // a[3]) for a in axes)
    heads, kvh, dim = case["heads"], case["kv_heads"], case["dim"]
    pairs = _pairs(case) * heads
    if case["op"] == "varlen":
        tok = otok = sum(_lengths(case))
    q, kv, out = tok * heads * dim * size, tok * kvh * dim * size, otok * heads * dim * size
    if case["op"] == "fused" and not case["grad"]:
        return {"bytes": q + 2 * kv + out, "flops": 4 * dim * pairs}
    # forward and backward: q, k, v and the output's gradient in, the output
    # and the gradients of q, k and v out
    total = {"bytes": 2 * (q + 2 * kv + out), "flops": 12 * dim * pairs}
    if case["op"] == "fused" and case["lse"]:
        total["bytes"] += otok * heads * size
    if case["op"] == "varlen":
        total["bytes"] += 4 * case["batch"] * case["extra"] * kvh * dim * size
    if case["op"] == "rpb":
        total["flops"] += 2 * pairs
        total["bytes"] += 2 * heads * math.prod(2 * a[1] - 1 for a in axes) * 4
    if case["op"] == "split":  # the weights are what this path is for
        total["bytes"] += pairs * size
    if case["op"] == "layer":  # input, output and their gradients; the weights
        c = heads * dim
        total["bytes"] = 4 * tok * c * size + 2 * (4 * c * c + 4 * c) * size
        total["flops"] += 3 * 2 * tok * 4 * c * c
    return total


def tolerance(case):
    """Relative error of another correct implementation (sums in another
    order; in 16 bits, intermediate values rounded at other points)."""
    if case["dtype"] == "f32":
        return {"rel": 2e-6, "max": 4e-5}
    if case["op"] in ("split", "layer"):  # weights and logits stored in 16 bits
        return {"rel": 2e-2, "max": 0.2} if case["dtype"] == "bf16" else {"rel": 3e-3, "max": 3e-2}
    return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 2e-2}


# ---------------------------------------------------------------------------

def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    axes = _axes(case)
    ext, osp = [a[0] for a in axes], [-(-a[0] // a[3]) for a in axes]
    n, heads, kvh, dim = case["batch"], case["heads"], case["kv_heads"], case["dim"]

    def normal(*shape, std=1.0, dtype=dt):
        return (torch.randn(shape, generator=g, device=DEVICE) * std).to(dtype)

    arg = {"kernel_size": tuple(a[1] for a in axes), "dilation": tuple(a[2] for a in axes)}
    s = {"case": case, "arg": arg}
    if case["op"] == "layer":
        c = heads * dim
        layer = natten_amd.NeighborhoodAttention2D(c, heads, **arg).to(DEVICE)
        with torch.no_grad():
            for p in layer.parameters():
                p.copy_(normal(*p.shape, std=0.02 if p.ndim == 1 else c ** -0.5,
                               dtype=torch.float32))
        s["layer"] = layer.to(dt)
        s["leaves"] = [normal(n, *ext, c).requires_grad_()] + list(layer.parameters())
        s["grad"] = normal(n, *ext, c)
        return s
    grad = case.get("grad", True)
    leaves = [normal(n, *ext, heads, dim), normal(n, *ext, kvh, dim), normal(n, *ext, kvh, dim)]
    if case["op"] == "varlen":
        order = torch.randperm(n, generator=torch.Generator().manual_seed(seed)).tolist()
        lens = _lengths(case)
        s["lens"] = torch.tensor([lens[i] for i in order], dtype=torch.int32)
        leaves += [normal(n, case["extra"], kvh, dim) for _ in range(2)]
    if case["op"] == "rpb":
        k, d = axes[0][1], axes[0][2]
        s["arg"] = {"kernel_size": k, "dilation": d}
        s["scale"] = dim ** -0.5
        leaves.append(normal(heads, *(2 * a[1] - 1 for a in axes), std=0.02))
    if grad:
        for t in leaves:
            t.requires_grad_()
        s["grad"] = normal(n, *osp, heads, dim)
    s["leaves"] = leaves
    return s


def run(s):
    case, arg, leaves = s["case"], s["arg"], s["leaves"]
    lse = None
    if case["op"] == "layer":
        out = s["layer"](leaves[0])
    elif case["op"] == "varlen":
        q, k, v, ek, ev = leaves
        out = natten_amd.na1d_varlen_gqa(q, k, v, s["lens"], additional_keys=ek,
                                         additional_values=ev, **arg)
    elif case["op"] == "split":
        q, k, v = leaves
        attn = torch.softmax(natten_amd.na2d_qk(q, k, **arg), dim=-1)
        out = natten_amd.na2d_av(attn, v, **arg)
    elif case["op"] == "rpb":
        q, k, v, rpb = leaves
        one = len(_axes(case)) == 1
        qk, av = ((allin1.na1d_qk_rpb, allin1.na1d_av_fused) if one else
                  (allin1.na2d_qk_rpb, allin1.na2d_av_fused))
        attn = torch.softmax(qk(q, k, rpb, scale=s["scale"], **arg), dim=-1)
        out = av(attn, v, **arg)
    else:
        axes = _axes(case)
        arg = dict(arg, stride=tuple(a[3] for a in axes), is_causal=tuple(a[4] for a in axes))
        out = FUSED[len(axes)](*leaves, return_lse=case["lse"], **arg)
        if case["lse"]:
            out, lse = out
    if not case.get("grad", True):
        return out
    grads = torch.autograd.grad(out, leaves, s["grad"])
    return [out, *([] if lse is None else [lse]), *grads]


# ---------------------------------------------------------------------------
# 64-bit values in plain torch

def _axis_keys(ext, k, d, s, ca):
    """Key positions [O, K] of each query of one axis, and whether they count:
    inside the query's dilation phase the window is centred on the query and
    moved back where it would leave the phase; a causal one ends at it."""
    p = torch.arange(0, ext, s)
    phase, i = p % d, p // d
    if ca:
        slot = (i - k + 1)[:, None] + torch.arange(k)
        return (phase[:, None] + d * slot.clamp(min=0)).to(DEVICE), (slot >= 0).to(DEVICE)
    size = (ext - phase + d - 1) // d
    start = torch.minimum((i - k // 2).clamp(min=0), size - k)
    pos = phase[:, None] + d * (start[:, None] + torch.arange(k))
    return pos.to(DEVICE), torch.ones_like(pos, dtype=torch.bool, device=DEVICE)


def _slots(axes):
    """Per slot, in row-major order: token of its key for each query, and
    whether it counts (None: always)."""
    pos, ok = zip(*(_axis_keys(*a) for a in axes))
    for flat in range(math.prod(a[1] for a in axes)):
        tok, good = torch.zeros((), dtype=torch.int64, device=DEVICE), None
        rest = []
        for a in reversed(axes):
            rest.append(flat % a[1])
            flat //= a[1]
        for a, p, o, j in zip(axes, pos, ok, reversed(rest)):
            tok = (tok[..., None] * a[0] + p[:, j]).reshape(-1)
            here = o[:, j]
            good = here if good is None else (good[:, None] & here).reshape(-1)
        yield tok, (None if bool(good.all()) else good)


def _window_attention(q, k, v, g, axes, scale, bias=None):
    """(out, lse, dq, dk, dv, dbias) of [tokens, heads, dim] float64 tensors
    of one sample; bias: (table [heads, cells], cell of (query, slot))."""
    axes = list(axes)
    toks = torch.zeros((), dtype=torch.int64, device=DEVICE)
    for ext, _, _, s, _ in axes:
        toks = (toks[..., None] * ext + torch.arange(0, ext, s, device=DEVICE)).reshape(-1)
    qs = q[toks]
    slots = list(_slots(axes))
    logits = []
    for j, (tok, ok) in enumerate(slots):
        x = (qs * k[tok]).sum(-1) * scale
        if bias is not None:
            x = x + bias[0][:, bias[1][:, j]].T
        logits.append(x if ok is None else x.masked_fill(~ok[:, None], -math.inf))
    logits = torch.stack(logits, -1)
    lse = torch.logsumexp(logits, -1)
    p = torch.exp(logits - lse[..., None])
    out = torch.zeros_like(qs)
    for j, (tok, _) in enumerate(slots):
        out += p[..., j, None] * v[tok]
    if g is None:
        return out, lse, None, None, None, None
    delta = (out * g).sum(-1)
    dqs, dk, dv = torch.zeros_like(qs), torch.zeros_like(k), torch.zeros_like(v)
    dbias = None if bias is None else torch.zeros_like(bias[0])
    for j, (tok, _) in enumerate(slots):
        ds = p[..., j] * ((g * v[tok]).sum(-1) - delta)
        dqs += scale * ds[..., None] * k[tok]
        dk.index_add_(0, tok, scale * ds[..., None] * qs)
        dv.index_add_(0, tok, p[..., j, None] * g)
        if bias is not None:
            dbias.index_add_(1, bias[1][:, j], ds.T.contiguous())
    dq = torch.zeros_like(q)
    dq[toks] = dqs
    return out, lse, dq, dk, dv, dbias


def _dense_attention(q, k, v, g, scale):
    """The same where every query sees every key, head by head."""
    parts = []
    for h in range(q.shape[1]):
        qh, kh, vh = (t[:, h].contiguous() for t in (q, k, v))
        x = qh @ kh.T.contiguous() * scale
        lse = torch.logsumexp(x, -1)
        p = torch.exp(x - lse[:, None])
        o = p @ vh
        if g is None:
            parts.append((o, lse))
            continue
        gh = g[:, h].contiguous()
        ds = p * (gh @ vh.T.contiguous() - (o * gh).sum(-1)[:, None])
        parts.append((o, lse, scale * (ds @ kh), scale * (ds.T.contiguous() @ qh),
                      p.T.contiguous() @ gh))
    got = [torch.stack(x, 1) for x in zip(*parts)]
    return (got + [None] * 4)[:6]


def _bias_cells(axes):
    """Cell of the bias table for each (query, slot): per axis the distance
    of key and query in dilation steps, moved to start at zero."""
    cell = torch.zeros(1, 1, dtype=torch.int64, device=DEVICE)
    for a in axes:
        pos, _ = _axis_keys(*a)
        off = (pos - torch.arange(0, a[0], a[3], device=DEVICE)[:, None]) // a[2] + a[1] - 1
        cell = (cell[:, None, :, None] * (2 * a[1] - 1) + off[None, :, None, :]).reshape(
            cell.shape[0] * off.shape[0], -1)
    return cell


def _varlen_exact(case, s):
    """Per sample: its own window attention over its own length, joined with
    the global tokens in one softmax; zero rows past its end."""
    q, k, v, ek, ev = (t.detach().double() for t in s["leaves"])
    g = s["grad"].double()
    (_, ks, d, _, _), rep = _axes(case)[0], case["heads"] // case["kv_heads"]
    scale = case["dim"] ** -0.5
    out, dq, dk, dv, dek, dev = (torch.zeros_like(t) for t in (q, q, k, v, ek, ev))
    for b, n in enumerate(s["lens"].tolist()):
        qb, gb = q[b, :n], g[b, :n]
        kb, vb, ekb, evb = (t.repeat_interleave(rep, 1)
                            for t in (k[b, :n], v[b, :n], ek[b], ev[b]))
        slots = [tok for tok, _ in _slots([(n, ks, d, 1, False)])]
        x = torch.stack([(qb * kb[tok]).sum(-1) * scale for tok in slots]
                        + [(qb * e).sum(-1) * scale for e in ekb], -1)
        p = torch.softmax(x, -1)
        o = torch.zeros_like(qb)
        for j, tok in enumerate(slots):
            o += p[..., j, None] * vb[tok]
        for j, e in enumerate(evb):
            o += p[..., len(slots) + j, None] * e
        delta = (o * gb).sum(-1)
        dqb, dkb, dvb = torch.zeros_like(qb), torch.zeros_like(kb), torch.zeros_like(vb)
        dekb, devb = torch.zeros_like(ekb), torch.zeros_like(evb)
        for j, tok in enumerate(slots):
            ds = scale * p[..., j] * ((gb * vb[tok]).sum(-1) - delta)
            dqb += ds[..., None] * kb[tok]
            dkb.index_add_(0, tok, ds[..., None] * qb)
            dvb.index_add_(0, tok, p[..., j, None] * gb)
        for j in range(ekb.shape[0]):
            w = p[..., len(slots) + j]
            ds = scale * w * ((gb * evb[j]).sum(-1) - delta)
            dqb += ds[..., None] * ekb[j]
            dekb[j] = (ds[..., None] * qb).sum(0)
            devb[j] = (w[..., None] * gb).sum(0)
        out[b, :n], dq[b, :n] = o, dqb
        for into, x in ((dk[b, :n], dkb), (dv[b, :n], dvb), (dek[b], dekb), (dev[b], devb)):
            into.copy_(x.reshape(x.shape[0], -1, rep, x.shape[-1]).sum(2))
    return [out, dq, dk, dv, dek, dev]


def _attention_exact(case, q, k, v, g, scale, bias=None):
    """(out, lse, dq, dk, dv, dbias) of [batch, *spatial, heads, dim]."""
    axes, rep = _axes(case), case["heads"] // case["kv_heads"]
    dense = all(a[1] >= a[0] and a[3] == 1 and not a[4] for a in axes)
    got = []
    for b in range(q.shape[0]):
        qb, kb, vb = (t[b].reshape(-1, *t.shape[-2:]) for t in (q, k, v))
        kb, vb = kb.repeat_interleave(rep, 1), vb.repeat_interleave(rep, 1)
        gb = None if g is None else g[b].reshape(-1, *g.shape[-2:])
        r = (_dense_attention(qb, kb, vb, gb, scale) if dense else
             _window_attention(qb, kb, vb, gb, axes, scale, bias))
        r = list(r)
        if g is not None:
            for i in (3, 4):
                r[i] = r[i].reshape(r[i].shape[0], -1, rep, r[i].shape[-1]).sum(2)
        got.append(r)
    osp = [-(-a[0] // a[3]) for a in axes]
    shapes = [(*osp, *q.shape[-2:]), (*osp, q.shape[-2]), q.shape[1:], k.shape[1:], v.shape[1:]]
    res = [None if got[0][i] is None else torch.stack([r[i] for r in got]).reshape(-1, *shapes[i])
           for i in range(5)]
    return (*res, None if got[0][5] is None else sum(r[5] for r in got))


def exact(case, seed):
    s = prepare(case, seed)
    with torch.no_grad():
        if case["op"] == "varlen":
            return _varlen_exact(case, s)
        scale = case["dim"] ** -0.5
        g = s["grad"].double() if "grad" in s else None
        if case["op"] == "layer":
            return _layer_exact(case, s, g, scale)
        q, k, v = (t.detach().double() for t in s["leaves"][:3])
        bias = None
        if case["op"] == "rpb":
            bias = (s["leaves"][3].detach().double().flatten(1), _bias_cells(_axes(case)))
        out, lse, dq, dk, dv, dbias = _attention_exact(case, q, k, v, g, scale, bias)
        if g is None:
            return out
        if bias is not None:
            return [out, dq, dk, dv, dbias.reshape(s["leaves"][3].shape)]
        return [out, *([lse] if case.get("lse") else []), dq, dk, dv]


def _layer_exact(case, s, g, scale):
    x = s["leaves"][0].detach().double()
    w = {n: p.detach().double() for n, p in s["layer"].named_parameters()}
    c, lead = x.shape[-1], x.shape[:-1]
    qkv = (x @ w["qkv.weight"].T + w["qkv.bias"]).reshape(*lead, 3, case["heads"], case["dim"])
    q, k, v = (t.contiguous() for t in qkv.unbind(-3))
    da = (g @ w["proj.weight"]).reshape(*lead, case["heads"], case["dim"])
    a, _, dq, dk, dv, _ = _attention_exact(case, q, k, v, da, scale)
    a = a.reshape(*lead, c)
    out = a @ w["proj.weight"].T + w["proj.bias"]
    dqkv = torch.stack([dq, dk, dv], -3).reshape(*lead, 3 * c)
    flat = lambda t: t.reshape(-1, t.shape[-1])  # noqa: E731
    grads = {"qkv.weight": flat(dqkv).T @ flat(x), "qkv.bias": flat(dqkv).sum(0),
             "proj.weight": flat(g).T @ flat(a), "proj.bias": flat(g).sum(0)}
    return [out, dqkv @ w["qkv.weight"], *(grads[n] for n in w)]
