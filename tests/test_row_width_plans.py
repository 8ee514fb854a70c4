"""Launches of middling size take rows of half or a quarter of the width: which, and that their results are those of any."""
import pytest
import torch

from helpers import TOL, assert_close, make_inputs, oracle_all, run_scan_with_grads
from quick_ssm_amd import _lib, hip_scan, scan

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
]


@pytest.mark.parametrize("shape,dtype,ahead,back", WIDTHS, ids=str)
def test_row_widths(shape, dtype, ahead, back):
    align = next(a for a in (8, 4, 2, 1) if shape[2] % a == 0)
    b = hip_scan.make_plan(*shape, dtype, dtype, _lib.QSSM_BACKWARD, align, 0, loose=True)
    f = hip_scan.make_plan(*shape, dtype, dtype, _lib.QSSM_FORWARD, align, b.ckpt_stride, loose=True)
    size = 4 if dtype is F32 else 2
    # (the forward's widest lanes take 16 bytes: the headline shape's rows of 32)
    assert (f.strip_cols * size, b.strip_cols * size) == (ahead, back)
    assert f.ckpt_stride == b.ckpt_stride and f.n_ckpt == b.n_ckpt


@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype", [((2, 1100, 384), BF), ((1, 2051, 512), F16), ((3, 1125, 361), BF), ((1, 4500, 256), BF),
                                         ((1, 4097, 256), F16), ((2, 1000, 320), F32), ((1, 700, 1728), F32), ((2, 300, 192), F16)],
                         ids=str)
def test_narrow_rows_match_the_oracle(gpu, shape, dtype):
    ops = make_inputs(shape, dtype, seed=shape[1])
    got, ref = run_scan_with_grads(scan, *ops, gpu), oracle_all(*ops)
    for name in ("y", "dx", "da", "db", "dc"):
        assert_close(name, got[name], ref[name], TOL[dtype])
