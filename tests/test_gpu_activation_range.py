"""The grouped kernels' activations (fp16 parts at one scale per token or per 64
intermediate columns) keep the width that their documents state, also far
below the largest value of their group.

Selections: K-quant matrices with a single weight 1 per row make the layer
out[t][h] = 64 x[t][1 + h % inter], through gate = 64 (silu(64) = 64 in fp32),
up = a column of x and down = a column of mid. Fewer than 64 tokens: three parts,
the result is exact for fp32 values within 2^38 of the largest. From 64 tokens
on two parts: each of the two roundings (x, mid) is at most 2^-23 relative for
values within 2^28 of the largest and, where the second part reaches fp16's
subnormals, 2^-18 (what two bf16 parts hold) within 2^33.

Wide rows: one column 2^16 to 2^30 above the others, in a block of zero weights,
every format: the fp32 bar against the oracle, rel-L2 <= 1e-5."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import oracle as O
import qw6_amd as Q
from qw6_amd import synth as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available(), "no GPU visible"
    c = Q.Context(0, max_tokens=128)
    yield c
    c.close()


def selection(q, rows, cols, pick):
    """Rows of a K-quant matrix whose only weight is 1, in column pick[r]."""
    bb = S.row_bytes(q, 256)
    m = np.zeros((rows, cols // 256, bb), np.uint8)
    one = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    if q == S.Q_Q6_K:   # q - 32 = 0: low nibbles 0, the two high bits 2
        m[:, :, 128:192] = 0xAA
    for r in range(rows):
        b, c = m[r, pick[r] // 256], pick[r] % 256
        sub, i = c // 32, c % 32
        if q == S.Q_Q6_K:
            b[208:210] = one
            b[192 + 2 * sub] = b[193 + 2 * sub] = 1
            b[64 * (sub // 4) + 32 * (sub % 2) + i] |= 1 << 4 * (sub % 4 // 2)   # 33
        else:
            b[0:2] = one
            if sub < 4:
                b[4 + sub] = 1
            else:
                b[12 + sub - 4] = 1
            b[(16 if q == S.Q_Q4_K_M else 48) + 32 * (sub // 2) + i] = 1 << 4 * (sub % 2)
    return m.reshape(-1)


class HostLayer:
    """A layer of given expert matrices [expert][gate, up, down] of (bytes, quant)."""

    def __init__(self, ctx, hidden, inter, mats):
        import torch
        self.mats, self.hidden, self.inter = mats, hidden, inter
        shapes = ((inter, hidden), (inter, hidden), (hidden, inter))
        self.keep = [[torch.from_numpy(np.ascontiguousarray(a)).cuda() for a, _ in m] for m in mats]
        self.table = ctx.experts(*[[(k[j].data_ptr(), m[j][1], *shapes[j]) for k, m in zip(self.keep, mats)]
                                   for j in range(3)])
        self.desc = Q.make_layer(hidden, inter, 1, self.table)

    def run(self, ctx, x, lg):
        import torch
        T = x.shape[0]
        out = torch.zeros(T, self.hidden, dtype=torch.float32, device="cuda")
        ctx.set_mode(2)
        try:
            ctx.moe_forward(self.desc, torch.from_numpy(x).cuda(), out, n_tok=T, logits=torch.from_numpy(lg).cuda())
            torch.cuda.synchronize()
        finally:
            ctx.set_mode(0)
        return out.cpu().numpy()


@pytest.mark.parametrize("gu,dn", [(S.Q_Q4_K_M, S.Q_Q6_K), (S.Q_Q6_K, S.Q_Q5_K), (S.Q_Q5_K, S.Q_Q4_K_M)])
def test_parts_hold_the_stated_width(ctx, gu, dn):
    hidden, inter = 512, 256
    rng = np.random.default_rng(91)
    pick_u = 1 + np.arange(inter)
    L = HostLayer(ctx, hidden, inter, [((selection(gu, inter, hidden, np.zeros(inter, int)), gu),
                                        (selection(gu, inter, hidden, pick_u), gu),
                                        (selection(dn, hidden, inter, np.arange(hidden) % inter), dn))] * 2)
    try:
        for T, low, bound in ((1, -30, 0.0), (17, -30, 0.0), (63, -30, 0.0),
                              (64, -20, 2.0 ** -22), (64, -25, 2.0 ** -17), (100, -25, 2.0 ** -17)):
            # full 24-bit mantissas, magnitudes 2^low .. 1 beside the largest, 2^6
            x = (1.0 + rng.random((T, hidden))) * 2.0 ** rng.integers(low, 0, (T, hidden)) * rng.choice([-1.0, 1.0], (T, hidden))
            x = x.astype(np.float32)
            x[:, 0] = 64.0
            lg = np.zeros((T, 2), np.float32)
            lg[:, 0] = rng.choice([1.0, -1.0], T) if T < 64 else 1.0   # two experts, or tiles of 32
            print("parts", gu, dn, T, low, flush=True)
            got = L.run(ctx, x, lg)
            want = 64.0 * x[:, 1 + np.arange(hidden) % inter]
            err = np.abs(got.astype(np.float64) - want) / np.abs(want)
            print("largest relative error %.3g" % err.max(), flush=True)
            assert err.max() <= bound, (T, low)
    finally:
        L.table.free()


FIELDS = {S.Q_Q4_K_M: (0, 2), S.Q_Q5_K: (0, 2), S.Q_Q6_K: (208,), S.Q_IQ2_XXS: (0,), S.Q_IQ2_S: (0,), S.Q_IQ3_S: (0,)}


@pytest.mark.parametrize("gu,dn", [(S.Q_Q4_K_M, S.Q_Q6_K), (S.Q_Q5_K, S.Q_Q5_K), (S.Q_Q6_K, S.Q_Q4_K_M),
                                   (S.Q_IQ2_XXS, S.Q_IQ3_S), (S.Q_IQ2_S, S.Q_IQ2_S), (S.Q_IQ3_S, S.Q_IQ2_XXS)])
def test_rows_of_wide_range(ctx, gu, dn):
    hidden, inter = 512, 256
    mats = []
    for e in range(2):
        m = [S.quant_matrix(92, 3 * e + k, q, r, c) for k, (q, r, c) in
             enumerate(((gu, inter, hidden), (gu, inter, hidden), (dn, hidden, inter)))]
        for a in m[:2]:   # the first block of every row: zero weights
            b = a.reshape(inter, hidden // 256, -1)
            for o in FIELDS[gu]:
                b[:, 0, o:o + 2] = 0
        mats.append(tuple((a, q) for a, q in zip(m, (gu, gu, dn))))
    L = HostLayer(ctx, hidden, inter, mats)
    ol = O.Layer(hidden, inter, 2, 1, None, mats, None)
    rng = np.random.default_rng(93)
    try:
        for T in (33, 64, 100):
            x = rng.normal(size=(T, hidden)).astype(np.float32)
            x[:, 5] = 2.0 ** np.array([16, 20, 24, 30])[np.arange(T) % 4]
            lg = rng.normal(size=(T, 2)).astype(np.float32)
            print("wide", gu, dn, T, flush=True)
            got = L.run(ctx, x, lg)
            rel = [cases.rel_l2(got[t], O.moe_layer(ol, x[t], logits=lg[t])[0]) for t in range(T)]
            print("rel-L2 max %.2e" % max(rel), flush=True)
            assert max(rel) <= 1e-5, (T, int(np.argmax(rel)))
    finally:
        L.table.free()
