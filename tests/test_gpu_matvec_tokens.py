"""Device matvec calls whose tokens do not fill the last workgroup's share: every
token against the oracle (the fp32 bar of the single-token calls), and nothing
written past the last."""
from __future__ import annotations

import numpy as np
import pytest

import cases
import oracle as O
import qw6_amd as Q
from qw6_amd import synth as S

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "no GPU visible"
    return torch


@pytest.fixture(scope="module")
def ctx(torch_dev):
    c = Q.Context(0, max_tokens=4)
    yield c
    c.close()


@pytest.mark.parametrize("rows,cols", [(70, 512), (70, 1280), (4096, 1280), (4096, 1536)])   # rows in LDS; any multiple of 256: one launch; two with a token over
@pytest.mark.parametrize("q", [S.Q_FP32, S.Q_Q4_K_M, S.Q_Q6_K, S.Q_IQ2_XXS, S.Q_IQ3_S])
def test_matvec_partial_shares(torch_dev, ctx, q, rows, cols):
    torch = torch_dev
    most = 33 if rows < 4096 else 9
    if q == S.Q_FP32:
        w = S.f32_normal(91, 1, rows * cols, 0.05).reshape(-1)
    else:
        w = S.quant_matrix(91, 1, q, rows, cols)
    dw = torch.from_numpy(np.ascontiguousarray(w)).cuda()
    xs = np.stack([S.f32_normal(92, 2 + t, cols, 1.0) for t in range(most)])
    dx = torch.from_numpy(xs).cuda()
    want = [O.matvec(q, w, rows, cols, xs[t]) for t in range(most)]
    for n in (1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 32, 33):
        if n > most:
            break
        y = torch.full((n + 1, rows), 7.0, dtype=torch.float32, device="cuda")
        print("matvec", q, rows, cols, n, flush=True)
        ctx.matvec((dw.data_ptr(), q, rows, cols), dx, y, n_tok=n)
        torch.cuda.synchronize()
        h = y.cpu().numpy()
        assert (h[n] == 7.0).all(), n
        for t in range(n):
            assert cases.rel_l2(h[t], want[t]) <= TOL, (n, t)
