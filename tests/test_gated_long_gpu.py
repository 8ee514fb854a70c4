"""Gated scans whose chains are cut into clusters of more than two tiles: few chains over a long sequence."""
import pytest
import torch

from helpers import TOL, assert_close
from quick_ssm_amd import _lib, gated_scan, hip_scan, scan
from quick_ssm_amd.gates import gate_prologue

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 2048, 1024), (1, 4100, 128), (2, 3001, 264), (1, 9000, 136)], ids=str)
@pytest.mark.parametrize("dtypes", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.float32, torch.float16),
                                    (torch.float32, torch.float32)], ids=str)
def test_matches_the_gate_pass_and_the_plain_scan(gpu, shape, dtypes):
    dtype, compute = dtypes
    B, L, S = shape
    plans = [gated_scan._plan(B, L, S, dtype, compute, dtype, d, 0, True) for d in (_lib.QSSM_FORWARD, _lib.QSSM_BACKWARD)]
    assert all(2 < p.cluster <= 8 for p in plans)
    gen = torch.Generator().manual_seed(L)
    pre = [torch.randn(shape, generator=gen) for _ in range(5)]
    pre[0] += 4.0                                   # decays near one: what crosses the tiles matters
    pre = [t.to(dtype).to(gpu).requires_grad_(True) for t in pre]
    dy = torch.randn(shape, generator=gen).to(dtype).to(gpu)
    y = gated_scan.gated_scan(*pre, compute_dtype=compute)
    got = [y, *torch.autograd.grad(y, pre, dy)]
    again = gated_scan.gated_scan(*pre, compute_dtype=compute)
    assert torch.equal(y, again) and hip_scan.workspace_status() == 0
    a, x, c, b = gate_prologue(*pre, compute)
    y2 = scan(x, a, b, c, out_dtype=dtype)
    want = [y2, *torch.autograd.grad(y2, pre, dy)]
    for name, g, w in zip(("y", "dA", "dB", "dCa", "dCb", "dD"), got, want):
        assert_close(name, g.detach().float().cpu(), w.detach().double().cpu().numpy(), TOL[compute])
