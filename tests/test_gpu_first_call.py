"""The first call of a context on a stream that does not wait for the default one:
the workspace it allocates is cleared before its kernels run, not under them."""
from __future__ import annotations

import pytest

import qw6_amd as Q
from qw6_amd import synth as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,T,hidden,inter", [(2, 2048, 256, 1024), (2, 2048, 2048, 512), (1, 16, 2048, 512)])
def test_first_call_on_a_side_stream(mode, T, hidden, inter):
    import torch

    from qw6_amd.workload import SynthLayer
    assert torch.cuda.is_available(), "no GPU visible"
    s = torch.cuda.Stream()
    x = torch.from_numpy(S.f32_normal(82, 1, T * hidden, 1.0).reshape(T, hidden)).cuda()
    lg = torch.from_numpy(S.f32_normal(82, 2, T * 16, 1.0).reshape(T, 16)).cuda()
    for turn in range(3):
        with Q.Context(0, max_tokens=T) as ctx:
            L = SynthLayer(ctx, 82, 0, "q4k", hidden=hidden, inter=inter, n_experts=16, top_k=4)
            try:
                ctx.set_mode(mode)
                first, again = torch.zeros_like(x), torch.zeros_like(x)
                torch.cuda.synchronize()
                print("first call, turn", turn, flush=True)
                for out in (first, again):
                    ctx.moe_forward(L.desc, x, out, n_tok=T, logits=lg, stream=s.cuda_stream)
                    torch.cuda.synchronize()
                assert torch.equal(first, again), turn
                assert bool(first.isfinite().all()) and float(first.abs().sum(1).min()) > 0.0
            finally:
                L.free()
