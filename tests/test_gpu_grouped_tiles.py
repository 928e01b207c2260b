"""The grouped kernels at the edges of their tiles: every expert sees exactly T
tokens, for T around the 4, 8, 16 and 32 entries of a tile's forms, over every format
and over row counts of one to eight blocks; and a call of more tokens than one
batch holds. Against the oracle, fp32 bar (rel-L2 <= 1e-5 per token): the
activations' fp16 parts hold 22 bits or more (1.2e-7 relative, once in gate/up and once
in down), the weights are exact, and sums of up to 2048 fp32 products, here and
in the oracle, stay below 2048 * 2^-24 / 16 = 8e-6 of the result's norm."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import oracle as O
import qw6_amd as Q

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "no GPU visible"
    return torch


@pytest.fixture(scope="module")
def ctx(torch_dev):
    c = Q.Context(0, max_tokens=128)
    yield c
    c.close()


def forward(torch, ctx, L, xs, lg, res=None):
    T = xs.shape[0]
    dx, dl = torch.from_numpy(xs).cuda(), torch.from_numpy(lg).cuda()
    dr = None if res is None else torch.from_numpy(res).cuda()
    out = torch.zeros(T, L.hidden, dtype=torch.float32, device="cuda")
    idx = torch.zeros(T, L.top_k, dtype=torch.int32, device="cuda")
    w = torch.zeros(T, L.top_k, dtype=torch.float32, device="cuda")
    ctx.set_mode(2)
    try:
        ctx.moe_forward(L.desc, dx, out, n_tok=T, logits=dl, residual=dr, idx=idx, w=w)
        torch.cuda.synchronize()
    finally:
        ctx.set_mode(0)
    return out.cpu().numpy(), idx.cpu().numpy(), w.cpu().numpy()


@pytest.mark.parametrize("hidden,inter", [(256, 256), (512, 1024), (2048, 2048)])
@pytest.mark.parametrize("mix", ["q4k", "q5k", "q6q4", "iq2a", "iq2b"])
def test_tile_edges_vs_oracle(torch_dev, ctx, mix, hidden, inter):
    from qw6_amd.workload import SynthLayer
    E = 4
    L = SynthLayer(ctx, 47, 0, mix, hidden=hidden, inter=inter, n_experts=E, top_k=E)
    try:
        ol = O.Layer(hidden, inter, E, E, None, [L.expert_host(e) for e in range(E)], L.shared_host())
        big = 73 if hidden < 2048 else 33
        xs = np.stack([cases.token_x(47, 6, t, hidden=hidden) for t in range(big)])
        lg = np.random.default_rng(47).normal(size=(big, E)).astype(np.float32)
        want = [O.moe_layer(ol, xs[t], logits=lg[t], nthreads=8) for t in range(big)]
        for T in (1, 4, 5, 8, 9, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 72, 73):
            if T > big:
                break
            print("tiles", mix, hidden, inter, T, flush=True)
            out, idx, w = forward(torch_dev, ctx, L, xs[:T], lg[:T])
            for t in range(T):
                oo, oi, ow = want[t]
                assert np.array_equal(idx[t], oi), (T, t)
                assert cases.rel_l2(out[t], oo) <= TOL, (T, t)
    finally:
        L.free()


def test_more_tokens_than_a_batch(torch_dev):
    """65536 tokens make a batch of the grouped kernels, whose sort takes 8192 tokens of
    top-2 a pass: tokens on both sides of every pass and batch of a longer call
    (given logits, residual) against the same tokens on their own."""
    from qw6_amd.workload import SynthLayer
    T, n, hidden = 65536 + 37, 64, 256
    with Q.Context(0, max_tokens=T) as c:
        L = SynthLayer(c, 48, 0, "q4k", hidden=hidden, inter=256, n_experts=4, top_k=2)
        try:
            rng = np.random.default_rng(48)
            xs = rng.normal(size=(T, hidden)).astype(np.float32)
            lg = rng.normal(size=(T, 4)).astype(np.float32)
            res = rng.normal(size=(T, hidden)).astype(np.float32)
            print("tokens", T, flush=True)
            out, idx, w = forward(torch_dev, c, L, xs, lg, res)
            for a in (0, *range(8192 - n // 2, T - n, 8192), T - n):
                o, i, v = forward(torch_dev, c, L, xs[a:a + n], lg[a:a + n], res[a:a + n])
                assert np.array_equal(idx[a:a + n], i) and np.array_equal(w[a:a + n], v)
                assert np.array_equal(out[a:a + n], o)   # a result depends on its own row only
        finally:
            L.free()
