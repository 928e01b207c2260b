"""The measured work of this framework: what a program built on it runs, at
the sizes it runs it, through the public entry points of qw6_amd.

listed() are the fixed cases, draw(rng) more of the same ranges. A case is a
dict of plain values; its "kind" names the entry point:

  matvec  Context.matvec: y[t] = deq(W) x[t], one resident GGUF matrix
  moe     Context.moe_forward: one routed-expert FFN layer over n_tok tokens,
          the router on the device, as a decoder layer calls it (post-attention
          norm fused in, residual added, the shared expert behind its gate)
  head    Context.output_greedy: final norm, vocabulary projection, argmax
  stack   one token through consecutive layers, the hidden state in place

Shapes are those of this repository's bench, tests and smoke check (hidden
2048, expert width 512, 256 experts of which 8 are selected, a 248,320-row
Q6_K head, 40 layers) and generic ones. Weights are seeded random GGUF blocks
whose scales give weights of about 0.02; hidden states are normal with a few
large channels and a common direction that the router's rows also have a
share of, so that experts are selected unevenly, as they are in a model.
"""
from __future__ import annotations

import math
import re
import weakref
from pathlib import Path

import numpy as np
import torch

import qw6_amd as Q

DEV = "cuda"
EPS = 1e-6
MAX_TOKENS = 2048

# GGUF formats: quant id, bytes per 256-weight block, fp16 scale fields as
# (byte offset, typical value): the values give weights of about 0.02.
FORMATS = {
    "q4k": (Q.Q_Q4_K_M, 144, ((0, 8e-5), (2, 6e-4))),
    "q5k": (Q.Q_Q5_K, 176, ((0, 4e-5), (2, 6.2e-4))),
    "q6k": (Q.Q_Q6_K, 210, ((208, 1.5e-5),)),
    "iq2xxs": (Q.Q_IQ2_XXS, 66, ((0, 4e-4),)),
    "iq2s": (Q.Q_IQ2_S, 82, ((0, 4e-4),)),
    "iq3s": (Q.Q_IQ3_S, 110, ((0, 1.5e-4),)),
}
# Layer mixes: formats of the routed gate/up, of the downs (by expert index,
# in turn), and of the shared expert's gate/up and down.
MIXES = {
    "q4k": ("q4k", ("q6k",), "q4k", "q6k"),
    "iq2m": ("iq2xxs", ("iq3s", "iq2s"), "q4k", "q6k"),
    "q5k": ("q5k", ("q5k",), "q5k", "q5k"),
    "q6q4": ("q6k", ("q4k",), "q6k", "q4k"),
    "iq2a": ("iq2xxs", ("iq3s",), "q4k", "q6k"),
    "iq2b": ("iq2s", ("iq2s",), "iq3s", "iq2xxs"),
}


def _moe(name, mix, n_tok, hidden=2048, inter=512, experts=256, top_k=8, norm=True, residual=True,
         shared=True, gate=True):
    return {"name": name, "kind": "moe", "mix": mix, "n_tok": n_tok, "hidden": hidden, "inter": inter,
            "experts": experts, "top_k": top_k, "norm": norm, "residual": residual, "shared": shared,
            "gate": gate}


def listed():
    return [
        # one quantized projection of one token: the smallest call, all latency
        {"name": "matvec_q4k_512x2048", "kind": "matvec", "fmt": "q4k", "rows": 512, "cols": 2048, "n_tok": 1},
        # a projection of a few drafted tokens, a width outside the layer kernels' set
        {"name": "matvec_q6k_1000x1280_t6", "kind": "matvec", "fmt": "q6k", "rows": 1000, "cols": 1280, "n_tok": 6},
        # decode: one token through one layer, both of the model's quant mixes
        _moe("decode_q4k", "q4k", 1),
        _moe("decode_iq2m", "iq2m", 1),
        # multi-token prediction: a token and its draft verified together
        _moe("mtp_q4k_t2", "q4k", 2),
        # a few sequences decoded as one batch
        _moe("batch_iq2m_t11", "iq2m", 11),
        # a short prompt, or a long draft verified
        _moe("verify_q4k_t33", "q4k", 33),
        # prefill of the usual chunk, and of a chunk that is no multiple of a tile
        _moe("prefill_q4k_t512", "q4k", 512),
        _moe("prefill_iq2m_t509", "iq2m", 509),
        # prefill of a long prompt in one call
        _moe("prefill_q4k_t2048", "q4k", 2048),
        # the next token: final norm, vocabulary projection, argmax
        {"name": "head_q6k", "kind": "head", "fmt": "q6k", "vocab": 248320, "hidden": 2048, "norm": True},
        # a decode step's FFN blocks through all layers of the model
        {"name": "stack_iq2m_40", "kind": "stack", "mix": "iq2m", "layers": 40, "hidden": 2048, "inter": 512,
         "experts": 256, "top_k": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    u = rng.random()
    if u < 0.2:
        fmt = rng.choice(sorted(FORMATS))
        return {"kind": "matvec", "fmt": fmt, "rows": _log(rng, 64, 8192), "cols": 256 * _log(rng, 1, 16),
                "n_tok": _log(rng, 1, 32)}
    if u < 0.3:
        return {"kind": "head", "fmt": rng.choice(["q6k", "q6k", "q4k", "q5k"]),
                "vocab": 32 * _log(rng, 1000, 7760), "hidden": rng.choice([1024, 2048, 2048]),
                "norm": rng.random() < 0.8}
    hidden, inter = rng.choice([(2048, 512)] * 6 + [(1024, 256), (1024, 512), (2048, 256), (512, 1024)])
    experts, top_k = rng.choice([(256, 8)] * 5 + [(64, 8), (128, 6), (64, 4)])
    shared = rng.random() < 0.85
    return {"kind": "moe", "mix": rng.choice(["q4k", "q4k", "iq2m", "iq2m"] + sorted(MIXES)),
            "n_tok": _log(rng, 1, MAX_TOKENS), "hidden": hidden, "inter": inter, "experts": experts,
            "top_k": top_k, "norm": rng.random() < 0.8, "residual": rng.random() < 0.8, "shared": shared,
            "gate": shared and rng.random() < 0.7}


# ---- inputs ---------------------------------------------------------------------

def _gen(seed, *ids):
    g = torch.Generator(device=DEV)
    h = seed & 0xFFFFFFFF
    for i in ids:
        h = (h * 1000003 + i + 12345) & 0xFFFFFFFFFFFF
    g.manual_seed(h)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _blocks(g, fmt, n):
    """n random GGUF blocks, uint8 [n, block bytes]."""
    _, bb, fields = FORMATS[fmt]
    b = torch.randint(0, 256, (n, bb), generator=g, device=DEV, dtype=torch.uint8)
    for off, value in fields:
        d = (value * (0.5 + torch.rand(n, generator=g, device=DEV))).to(torch.float16)
        b[:, off:off + 2] = d.view(torch.uint8).reshape(n, 2)
    return b


def _matrix(g, fmt, rows, cols):
    """A resident GGUF matrix: its bytes, 16-byte aligned (a torch allocation)."""
    return _blocks(g, fmt, rows * (cols // 256)).reshape(-1)


def _desc(buf, fmt, rows, cols, offset=0):
    return (buf.data_ptr() + offset, FORMATS[fmt][0], rows, cols)


_context = None


def _ctx():
    """The one context that a program keeps."""
    global _context
    if _context is None:
        _context = Q.Context(0, max_tokens=MAX_TOKENS)
    return _context


class Layer:
    """The resident weights of one MoE layer and its expert table."""

    def __init__(self, seed, mix, hidden, inter, experts, top_k, norm=True, shared=True, gate=True):
        g = _gen(seed, 1)
        gu, downs, sgu, sdn = MIXES[mix]
        self.hidden, self.inter, self.n, self.top_k = hidden, inter, experts, top_k
        self.fmt = [(gu, gu, downs[e % len(downs)]) for e in range(experts)]
        shapes = ((inter, hidden), (inter, hidden), (hidden, inter))
        self.shapes = shapes
        self.packs, self.offs, mats = [], [], []
        for k, (r, c) in enumerate(shapes):
            fmts = [f[k] for f in self.fmt]
            size = {f: (r * (c // 256) * FORMATS[f][1] + 255) // 256 * 256 for f in set(fmts)}
            offs = np.concatenate([[0], np.cumsum([size[f] for f in fmts])]).tolist()
            buf = torch.zeros(offs[-1], dtype=torch.uint8, device=DEV)
            if len(size) == 1:   # one format: the whole pack at once
                f, n = fmts[0], r * (c // 256) * FORMATS[fmts[0]][1]
                v = buf.view(experts, size[f])
                for e0 in range(0, experts, 64):
                    m = min(64, experts - e0)
                    v[e0:e0 + m, :n] = _blocks(g, f, m * r * (c // 256)).view(m, n)
            else:
                for e in range(experts):
                    b = _matrix(g, fmts[e], r, c)
                    buf[offs[e]:offs[e] + b.numel()] = b
            self.packs.append(buf)
            self.offs.append(offs)
            mats.append([_desc(buf, fmts[e], r, c, offs[e]) for e in range(experts)])
        self.dir = _normal(_gen(seed, 2), hidden)
        self.dir /= self.dir.norm()
        self.router = 0.02 * _normal(g, experts, hidden)
        self.router += (0.5 * _normal(g, experts, 1)) * self.dir / (0.2 * math.sqrt(hidden))
        self.shared = None
        if shared:
            fm = (sgu, sgu, sdn)
            self.shared = [(_matrix(g, fm[k], *shapes[k]), fm[k]) for k in range(3)]
        self.gate = 0.02 * _normal(g, hidden) if gate and shared else None
        self.norm = 1.0 + 0.1 * _normal(g, hidden) if norm else None
        self.table = _ctx().experts(*mats)
        weakref.finalize(self, self.table.free)
        self.desc = Q.make_layer(
            hidden, inter, top_k, self.table, router=self.router, shared_router=self.gate,
            norm_w=self.norm, norm_eps=EPS,
            shared=None if not shared else [_desc(b, f, *shapes[k]) for k, (b, f) in enumerate(self.shared)])

    def matrix(self, e, k):
        """Bytes and format of matrix k of expert e (e == n: the shared expert)."""
        if e == self.n:
            return self.shared[k]
        f = self.fmt[e][k]
        r, c = self.shapes[k]
        o = self.offs[k][e]
        return self.packs[k][o:o + r * (c // 256) * FORMATS[f][1]], f


def _hidden_states(g, direction, n, hidden):
    x = _normal(g, n, hidden)
    cols = torch.randint(0, hidden, (4,), generator=g, device=DEV)
    x[:, cols] *= 8.0
    return x + 0.2 * math.sqrt(hidden) * direction


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _tokens(seed, layer, n):
    """n hidden states none of whose first top_k + 1 router logits are within
    1e-4 of each other, so that every correct implementation selects the same
    experts in the same order."""
    g = _gen(seed, 3)
    keep, have = [], 0
    while have < n:
        x = _hidden_states(g, layer.dir, n + n // 16 + 16, layer.hidden)
        xd = x.double()
        lg = (_rms(xd, layer.norm.double()) if layer.norm is not None else xd) @ layer.router.double().t()
        top = lg.topk(layer.top_k + 1, dim=1).values
        x = x[(top[:, :-1] - top[:, 1:]).min(dim=1).values > 1e-4]
        keep.append(x)
        have += x.shape[0]
    return torch.cat(keep)[:n].contiguous()


class State:
    pass


def prepare(case, seed):
    s = State()
    s.case, s.ctx = case, _ctx()
    kind = case["kind"]
    if kind == "matvec":
        g = _gen(seed, 4)
        s.W = _matrix(g, case["fmt"], case["rows"], case["cols"])
        s.w = _desc(s.W, case["fmt"], case["rows"], case["cols"])
        s.x = _normal(g, case["n_tok"], case["cols"])
        s.y = torch.empty(case["n_tok"], case["rows"], dtype=torch.float32, device=DEV)
    elif kind == "moe":
        s.layer = Layer(seed, case["mix"], case["hidden"], case["inter"], case["experts"], case["top_k"],
                        case["norm"], case["shared"], case["gate"])
        T = case["n_tok"]
        s.x = _tokens(seed, s.layer, T)
        s.res = 0.1 * _normal(_gen(seed, 5), T, case["hidden"]) if case["residual"] else None
        s.out = torch.empty_like(s.x)
        s.idx = torch.empty(T, case["top_k"], dtype=torch.int32, device=DEV)
        s.w = torch.empty(T, case["top_k"], dtype=torch.float32, device=DEV)
    elif kind == "head":
        g = _gen(seed, 6)
        s.W = _matrix(g, case["fmt"], case["vocab"], case["hidden"])
        s.w = _desc(s.W, case["fmt"], case["vocab"], case["hidden"])
        s.x = _normal(g, case["hidden"])
        s.norm = 1.0 + 0.1 * _normal(g, case["hidden"]) if case["norm"] else None
        s.logits = torch.empty(case["vocab"], dtype=torch.float32, device=DEV)
        s.token = torch.empty(1, dtype=torch.int32, device=DEV)
    else:
        s.layers = [Layer(seed + 7919 * l, case["mix"], case["hidden"], case["inter"], case["experts"],
                          case["top_k"]) for l in range(case["layers"])]
        s.x = _hidden_states(_gen(seed, 7), s.layers[0].dir, 1, case["hidden"])
        s.h = torch.empty_like(s.x)
        s.idx = torch.empty(case["layers"], case["top_k"], dtype=torch.int32, device=DEV)
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "matvec":
        s.ctx.matvec(s.w, s.x, s.y, n_tok=s.case["n_tok"])
        return s.y
    if kind == "moe":
        s.ctx.moe_forward(s.layer.desc, s.x, s.out, n_tok=s.case["n_tok"], residual=s.res, idx=s.idx, w=s.w)
        return {"out": s.out, "idx": s.idx, "w": s.w}
    if kind == "head":
        s.ctx.output_greedy(s.w, s.x, s.logits, s.token, norm_w=s.norm, eps=EPS)
        return {"logits": s.logits, "token": s.token}
    src = s.x
    for l, layer in enumerate(s.layers):
        s.ctx.moe_forward(layer.desc, src, s.h, n_tok=1, residual=src, idx=s.idx[l])
        src = s.h
    return s.h


# ---- what a pass cannot do without -----------------------------------------------------

def _bytes(fmt, rows, cols):
    return rows * (cols // 256) * FORMATS[fmt][1]


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        r, c, t = case["rows"], case["cols"], case["n_tok"]
        return {"bytes": _bytes(case["fmt"], r, c) + 4 * t * (r + c), "flops": 2 * r * c * t}
    if kind == "head":
        r, c = case["vocab"], case["hidden"]
        return {"bytes": _bytes(case["fmt"], r, c) + 4 * (r + 2 * c) + 4, "flops": 2 * r * c}
    H, I, E, k = case["hidden"], case["inter"], case["experts"], case["top_k"]
    T = 1 if kind == "stack" else case["n_tok"]
    gu, downs, sgu, sdn = MIXES[case["mix"]]
    # distinct experts that T tokens' selections reach, drawn evenly
    distinct = E * (1.0 - (1.0 - k / E) ** T)
    dn = sum(_bytes(f, H, I) for f in downs) / len(downs)
    weights = distinct * (2 * _bytes(gu, I, H) + dn) + 4 * E * H
    n = k
    if kind == "stack" or case["shared"]:
        weights += 2 * _bytes(sgu, I, H) + _bytes(sdn, H, I)
        n += 1
    io = 4 * T * H * (3 if kind == "stack" or case["residual"] else 2) + 8 * T * k
    flops = 2 * T * (n * 3 * H * I + E * H)
    layers = case["layers"] if kind == "stack" else 1
    return {"bytes": int(layers * (weights + io)), "flops": int(layers * flops)}


def tolerance(case):
    # About four times the largest error against exact() that was measured:
    # 2.6e-7 for the layer on the fp32 kernels and 3e-6 to 4.6e-6 on the
    # grouped ones (16 tokens and more), 2.6e-6 for the head, whose products
    # take 16 significant bits of the activations, 1.7e-7 for one matrix.
    if case["kind"] == "moe":
        return {"rel": 2e-5 if case["n_tok"] >= 16 else 2e-6}
    return {"rel": {"head": 1e-5, "matvec": 1e-6, "stack": 5e-6}[case["kind"]]}


# ---- the same in 64 bits -----------------------------------------------------------------

_grids = None


def _tables():
    """The IQ formats' lattice points, from the packed table this repository's
    formats are defined by (a data file: 2 or 3 bits per value)."""
    global _grids
    if _grids is None:
        text = (Path(Q.__file__).resolve().parent / "csrc" / "iq_grid_data.h").read_text()
        codes = {m.group(1): [int(v, 16) for v in re.findall(r"0x[0-9a-fA-F]+", m.group(2))]
                 for m in re.finditer(r"qw6_(iq\w+)_codes\[\d+\] = \{(.*?)\};", text, re.S)}
        level = (8.0, 25.0, 43.0, 43.0)
        _grids = {
            "iq2xxs": [[level[(c >> 2 * j) & 3] for j in range(8)] for c in codes["iq2xxs"]],
            "iq2s": [[level[(c >> 2 * j) & 3] for j in range(8)] for c in codes["iq2s"]],
            "iq3s": [[2.0 * ((c >> 3 * j) & 7) + 1.0 for j in range(4)] for c in codes["iq3s"]],
        }
        _grids = {k: torch.tensor(v, dtype=torch.float64, device=DEV) for k, v in _grids.items()}
    return _grids


def _dequant(buf, fmt, rows, cols):
    """A GGUF matrix in float64, [rows, cols]."""
    bb = FORMATS[fmt][1]
    b = buf.view(-1, bb)
    n = b.shape[0]
    i = b.to(torch.int64)

    def half(off):
        return b[:, off:off + 2].contiguous().view(torch.float16).double()

    def bits(v, shifts, mask):
        return (v.unsqueeze(-1) >> torch.tensor(shifts, device=DEV)) & mask

    if fmt in ("q4k", "q5k"):
        d, dmin, s = half(0), half(2), i[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = i[:, bb - 128:].view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32)
        if fmt == "q5k":
            q = q | (bits(i[:, 16:48], range(8), 1).transpose(1, 2) << 4)
        w = (d * sc).unsqueeze(-1) * q - (dmin * mn).unsqueeze(-1)
    elif fmt == "q6k":
        ql, qh = i[:, :128].view(n, 2, 2, 32), i[:, 128:192].view(n, 2, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)                      # runs k = 0 .. 3
        hi = bits(qh, (0, 2, 4, 6), 3).permute(0, 1, 3, 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(n, 8, 2)[:, :, 0]   # the even scale of a 32-run
        w = (half(208) * sc).unsqueeze(-1) * ((lo | (hi << 4)) - 32).view(n, 8, 32)
    else:
        grid = _tables()[fmt]
        d = half(0)
        if fmt == "iq2xxs":
            p = i[:, 2:66].view(n, 8, 8)
            aux = p[:, :, 4] | (p[:, :, 5] << 8) | (p[:, :, 6] << 16) | (p[:, :, 7] << 24)
            s7 = bits(aux, (0, 7, 14, 21), 127)
            par = bits(s7, range(7), 1).sum(-1) & 1
            v, sg = grid[p[:, :, :4]], s7 | (par << 7)
            db = (d * (0.5 + (aux >> 28)) * 0.25).unsqueeze(-1)
        elif fmt == "iq2s":
            hi = bits(i[:, 66:74], (0, 2, 4, 6), 3)
            v, sg = grid[i[:, 2:34].view(n, 8, 4) | (hi << 8)], i[:, 34:66].view(n, 8, 4)
            db = (d * (0.5 + bits(i[:, 74:82], (0, 4), 15).view(n, 16)) * 0.25).view(n, 8, 2).repeat_interleave(2, -1)
        else:
            hi = bits(i[:, 66:74], range(8), 1)
            v = grid[i[:, 2:66].view(n, 8, 8) | (hi << 8)].view(n, 8, 4, 8)
            sg = i[:, 74:106].view(n, 8, 4)
            db = (d * (1 + 2 * bits(i[:, 106:110], (0, 4), 15).view(n, 8))).unsqueeze(-1)
        w = db.unsqueeze(-1) * v * (1.0 - 2.0 * bits(sg, range(8), 1))
    return w.reshape(rows, cols)


def _exact_moe(layer, x, residual):
    """(out, idx, w) of one layer in 64 bits."""
    x = x.double()
    xin = _rms(x, layer.norm.double()) if layer.norm is not None else x
    val, idx = (xin @ layer.router.double().t()).topk(layer.top_k, dim=1)
    w = torch.softmax(val, dim=1)
    H, I = layer.hidden, layer.inter

    def ffn(e, rows):
        g, u, dn = (_dequant(*layer.matrix(e, k), *layer.shapes[k]) for k in range(3))
        a = rows @ g.t()
        return (a * torch.sigmoid(a) * (rows @ u.t())) @ dn.t()

    out = torch.zeros(x.shape[0], H, dtype=torch.float64, device=DEV)
    for e in idx.unique().tolist():
        t, k = (idx == e).nonzero(as_tuple=True)
        out.index_add_(0, t, w[t, k].unsqueeze(-1) * ffn(e, xin[t]))
    if layer.shared is not None:
        y = ffn(layer.n, xin)
        out += y if layer.gate is None else torch.sigmoid(xin @ layer.gate.double()).unsqueeze(-1) * y
    if residual is not None:
        out += residual.double()
    return out, idx, w


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "matvec":
        return s.x.double() @ _dequant(s.W, case["fmt"], case["rows"], case["cols"]).t()
    if kind == "moe":
        out, idx, w = _exact_moe(s.layer, s.x, s.res)
        return {"out": out, "idx": idx.to(torch.int32), "w": w}
    if kind == "head":
        r, c, step = case["vocab"], case["hidden"], 32 * 512
        x = s.x.double()
        if s.norm is not None:
            x = _rms(x, s.norm.double())
        rb = (c // 256) * FORMATS[case["fmt"]][1]
        lg = torch.cat([_dequant(s.W[r0 * rb:min(r, r0 + step) * rb], case["fmt"], min(r, r0 + step) - r0, c) @ x
                        for r0 in range(0, r, step)])
        return {"logits": lg, "token": lg.argmax().reshape(1).to(torch.int32)}
    h = s.x
    for layer in s.layers:
        h = _exact_moe(layer, h, h)[0]
    return h
