"""The batched path's router logits (calls without given logits) against 64-bit
sums, through the routing results that moe_forward returns: calls just above
the size from which the matrix kernel forms them, both of its tile sizes, every
hidden size, tokens and experts that leave partial tiles."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import oracle as O
import qw6_amd as Q

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "no GPU visible"
    return torch


@pytest.mark.parametrize("hidden,n_experts,T", [
    (256, 64, 161), (512, 100, 103), (1024, 96, 107), (2048, 256, 40), (2048, 256, 41),   # 40: one wave per expert
    (2048, 256, 512), (2048, 256, 513), (256, 100, 1313)])                                # 16 x 16, then 32 x 32
def test_router_logits_vs_float64(torch_dev, hidden, n_experts, T):
    torch = torch_dev
    from qw6_amd.workload import SynthLayer
    with Q.Context(0, max_tokens=T) as ctx:
        L = SynthLayer(ctx, 43, 0, "q4k", hidden=hidden, inter=256, n_experts=n_experts, top_k=8)
        try:
            xs = np.stack([cases.token_x(43, 5, t, hidden=hidden) for t in range(T)])
            dx = torch.from_numpy(xs).cuda()
            dout = torch.zeros(T, hidden, dtype=torch.float32, device="cuda")
            didx = torch.zeros(T, 8, dtype=torch.int32, device="cuda")
            dw = torch.zeros(T, 8, dtype=torch.float32, device="cuda")
            print("router", hidden, n_experts, T, flush=True)
            ctx.set_mode(2)
            ctx.moe_forward(L.desc, dx, dout, n_tok=T, idx=didx, w=dw)
            torch.cuda.synchronize()
            idx, w = didx.cpu().numpy(), dw.cpu().numpy()
            router = L.router_host().reshape(n_experts, hidden)
        finally:
            L.free()
    lg = xs.astype(np.float64) @ router.astype(np.float64).T
    # A product passes at most 4 roundings in its MFMA, 3 + 8 + 3 in the sums after it
    # (k_pre_router: 32 + 6), its own included; one more for the oracle's fp32 logits.
    bound = 40 * 2.0 ** -24 * (np.abs(xs).astype(np.float64) @ np.abs(router).astype(np.float64).T).max(1)
    compared = 0
    for t in range(T):
        top = np.sort(lg[t])[::-1][:9]
        if (top[:-1] - top[1:]).min() <= 2 * bound[t]:
            continue   # either order is right
        oi, ow = O.moe_route(lg[t].astype(np.float32), 8)
        assert np.array_equal(idx[t], oi), t
        # a weight is a ratio of exponentials: relative error 2 bound, and the fp32 exponentials'
        assert np.abs(w[t] - ow).max() <= 2 * bound[t] + 2e-5, t
        compared += 1
    assert compared >= 0.9 * T
