"""Launches of middling size take rows of half or a quarter of the width: which, and that their results are those of any."""
import pytest
import torch

from helpers import TOL, assert_close, make_inputs, oracle_all, run_scan_with_grads
from quick_ssm_amd import _lib, gated_scan, hip_scan, scan
from quick_ssm_amd.gates import gate_prologue

BF, F16, F32 = torch.bfloat16, torch.float16, torch.float32
# (shape, storage): bytes of a row piece forward and backward
WIDTHS = [
    ((8, 4096, 2048), BF, 512, 512),      # large: the wider pieces stream faster
    ((6, 7480, 384), BF, 256, 256),       # one and a half strips of 512 bytes
    ((2, 8192, 512), F16, 256, 256),      # few chains over a long sequence
    ((8, 2048, 1024), BF, 512, 512),      # neither
    ((13, 1125, 361), BF, 256, 512),      # rows that end anywhere
    ((34, 3335, 152), F16, 512, 512),     # the same without less padding
    ((1, 21625, 256), BF, 128, 128),      # the chain is all there is
    ((1, 20000, 320), F32, 256, 256),
    ((4, 4096, 1024), F32, 512, 512),
    # rows off 128-byte lines, whose chains are shorter than the stream: padding alone does not pay
    ((4, 1019, 1976), F32, 512, 512),
    ((19, 638, 1616), BF, 512, 512),
    ((4, 7540, 1384), F16, 512, 512),
    ((5, 418, 928), F32, 128, 512),       # on them, and hardly a chain (the forward is short of tiles)
]


def _widths(shape, dtype):
    align = next(a for a in (8, 4, 2, 1) if shape[2] % a == 0)
    b = hip_scan.make_plan(*shape, dtype, dtype, _lib.QSSM_BACKWARD, align, 0, loose=True)
    f = hip_scan.make_plan(*shape, dtype, dtype, _lib.QSSM_FORWARD, align, b.ckpt_stride, loose=True)
    size = 4 if dtype is F32 else 2
    assert f.ckpt_stride == b.ckpt_stride and f.n_ckpt == b.n_ckpt
    return f.strip_cols * size, b.strip_cols * size


@pytest.mark.parametrize("shape,dtype,ahead,back", WIDTHS, ids=str)
def test_row_widths(shape, dtype, ahead, back):
    # (the forward's widest lanes take 16 bytes: the headline shape's rows of 32)
    assert _widths(shape, dtype) == (ahead, back)


# (shape, storage, compute): lanes of a row forward and backward
GATED = [
    ((4, 2100, 384), BF, BF, 32, 32),      # less padding, on 128-byte lines
    ((4, 4096, 1024), BF, BF, 32, 64),     # the forward's chain
    ((8, 4096, 1024), BF, BF, 64, 64),     # neither
    ((1, 7000, 856), BF, BF, 32, 64),      # off them: the forward alone, for its chain
    ((1, 6000, 944), F32, F16, 32, 64),
    ((20, 394, 856), BF, BF, 64, 64),      # off them and no such chain
    ((14, 615, 2952), F32, F16, 64, 64),
    ((1, 4852, 1840), BF, BF, 32, 64),
]


def _gated_plans(shape, dtype, compute):
    first = gated_scan._plan(*shape, dtype, compute, dtype, _lib.QSSM_BACKWARD, 0)
    f = gated_scan._plan(*shape, dtype, compute, dtype, _lib.QSSM_FORWARD, first.seg_len, True)
    b = gated_scan._plan(*shape, dtype, compute, dtype, _lib.QSSM_BACKWARD, f.ckpt_stride, True)
    # the backward that the states are saved for is the one that is launched
    assert b.seg_len == first.seg_len == f.ckpt_stride == b.ckpt_stride and f.seg_len % f.ckpt_stride == 0 and f.n_ckpt == b.n_ckpt
    return f, b


@pytest.mark.parametrize("shape,dtype,compute,ahead,back", GATED, ids=str)
def test_gated_row_widths(shape, dtype, compute, ahead, back):
    f, b = _gated_plans(shape, dtype, compute)
    assert (1 << f.g_log2, 1 << b.g_log2) == (ahead, back)


# Small launches, whose rows are narrow for want of tiles.
@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype", [((2, 1100, 384), BF), ((1, 2051, 512), F16), ((3, 1125, 361), BF), ((1, 4500, 256), BF),
                                         ((1, 4097, 256), F16), ((2, 1000, 320), F32), ((1, 700, 1728), F32), ((2, 300, 192), F16)],
                         ids=str)
def test_narrow_rows_match_the_oracle(gpu, shape, dtype):
    ops = make_inputs(shape, dtype, seed=shape[1])
    got, ref = run_scan_with_grads(scan, *ops, gpu), oracle_all(*ops)
    for name in ("y", "dx", "da", "db", "dc"):
        assert_close(name, got[name], ref[name], TOL[dtype])


# Launches with tiles enough for the full width: 512-lane forwards with rows of 256 bytes over saved states half a tile
# apart, narrow forwards over wider backwards, rows of 128 bytes in a backward, fp32.
@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype,ahead,back", [w for w in WIDTHS if min(w[2:]) < 512 and w[0][1] > 418], ids=str)
def test_rows_that_the_rule_narrows_match_the_oracle(gpu, shape, dtype, ahead, back):
    assert _widths(shape, dtype) == (ahead, back)
    ops = make_inputs(shape, dtype, seed=shape[1])
    got, ref = run_scan_with_grads(scan, *ops, gpu), oracle_all(*ops)
    assert hip_scan.workspace_status() == 0
    for name in ("y", "dx", "da", "db", "dc"):
        assert_close(name, got[name], ref[name], TOL[dtype])


@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype,compute,ahead,back", [w for w in GATED if min(w[3:]) < 64], ids=str)
def test_gated_rows_that_the_rule_narrows_match_the_gate_pass_and_the_scan(gpu, shape, dtype, compute, ahead, back):
    f, b = _gated_plans(shape, dtype, compute)
    assert (1 << f.g_log2, 1 << b.g_log2) == (ahead, back)
    gen = torch.Generator().manual_seed(shape[1])
    pre = [torch.randn(shape, generator=gen) for _ in range(5)]
    pre[0] += 4.0                                   # decays near one: what crosses the tiles matters
    pre = [t.to(dtype).to(gpu).requires_grad_(True) for t in pre]
    dy = torch.randn(shape, generator=gen).to(dtype).to(gpu)
    y = gated_scan.gated_scan(*pre, compute_dtype=compute)
    got = [y, *torch.autograd.grad(y, pre, dy)]
    assert hip_scan.workspace_status() == 0
    a, x, c, b = gate_prologue(*pre, compute)
    y2 = scan(x, a, b, c, out_dtype=dtype)
    want = [y2, *torch.autograd.grad(y2, pre, dy)]
    for name, g, w in zip(("y", "dA", "dB", "dCa", "dCb", "dD"), got, want):
        assert_close(name, g.detach().float().cpu(), w.detach().double().cpu().numpy(), TOL[compute])
