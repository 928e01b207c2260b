"""The batched path's workspace: on the CPU (tests/c/prefill_ws.cpp) its layout, its growth
over layers of different shapes and allocations that fail; on the GPU one context
that alternates two shapes neither of which holds the other."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
HIP_INC = Path("/opt/rocm/include")


@pytest.mark.skipif(shutil.which("g++") is None or not (HIP_INC / "hip").exists(), reason="needs g++ and the HIP headers")
def test_workspace_growth_and_failed_allocations(tmp_path):
    exe = tmp_path / "prefill_ws"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-isystem", str(HIP_INC),
                    "-I", str(ROOT / "include"), "-I", str(ROOT / "qw6_amd" / "csrc"), "-o", str(exe),
                    str(ROOT / "tests" / "c" / "prefill_ws.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


@pytest.mark.gpu
def test_alternating_shapes_keep_one_workspace():
    """Layers of 1024 x 256 and 256 x 1024 in turn through one context, the first calls on a
    stream that does not wait for the default one: results equal those of the
    per-token kernels, and after one call of each no call takes device memory."""
    import torch

    import cases
    import qw6_amd as Q
    from qw6_amd import synth as S
    from qw6_amd.workload import SynthLayer
    assert torch.cuda.is_available(), "no GPU visible"
    T = 2048
    with Q.Context(0, max_tokens=T) as ctx:
        runs = []
        for h, i in ((1024, 256), (256, 1024)):
            L = SynthLayer(ctx, 81, 0, "q4k", hidden=h, inter=i, n_experts=16, top_k=4)
            x = torch.from_numpy(S.f32_normal(81, h, T * h, 1.0).reshape(T, h)).cuda()
            lg = torch.from_numpy(S.f32_normal(81, 3, T * 16, 1.0).reshape(T, 16)).cuda()
            runs.append((L, x, lg, torch.empty_like(x), torch.empty_like(x)))
        s = torch.cuda.Stream()
        try:
            for L, x, lg, out, ref in runs:
                ctx.set_mode(1)
                ctx.moe_forward(L.desc, x, ref, n_tok=T, logits=lg)
            ctx.set_mode(2)
            torch.cuda.synchronize()
            free = None
            for turn in range(4):
                for L, x, lg, out, ref in runs:
                    out.zero_()
                    torch.cuda.synchronize()
                    with torch.cuda.stream(s):
                        ctx.moe_forward(L.desc, x, out, n_tok=T, logits=lg, stream=s.cuda_stream)
                    torch.cuda.synchronize()
                    a, b = out.cpu().numpy(), ref.cpu().numpy()
                    assert max(cases.rel_l2(a[t], b[t]) for t in range(T)) <= 1e-5, (turn, L.hidden)
                now = torch.cuda.mem_get_info()[0]
                assert free is None or now == free, (turn, free, now)
                free = now
        finally:
            ctx.set_mode(0)
            for L, *_ in runs:
                L.free()
