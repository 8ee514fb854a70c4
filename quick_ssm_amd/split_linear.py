"""Linear maps of the SSM layer over fp32 parameters, on the 16-bit matrix cores (csrc/gemm_split.hip).

A layer with fp32 parameters spends nine tenths of its time in its projections (quick_ssm/layers.py:76-80,106): the
library's fp32 products run at the fp32 MFMA rate, a sixteenth of the fp16 one.  `qssm_split_gemm` takes every element
as the sum of two scaled fp16 values and accumulates three products in fp32, with an error at or below that of fp32
products.  Here is the rule for when it is used; maxima, scratch and the calls are in csrc/torch_scan.cpp, the autograd
functions that use them in quick_ssm_amd/layers.py.
"""
from __future__ import annotations

from typing import List, NamedTuple, Optional, Sequence, Tuple

import torch

from . import hip_scan

Tensor = torch.Tensor

# Multiply-adds (over all weights of a launch) below which the library's product stays, because the fixed costs of the
# maxima, the prologue, the sums over parts and their launches exceed the gain.  us for output, input gradient and weight
# gradient together, library against these: 4096 rows, 1024 x 256 (1.1e9) 79 against 129; 4096 rows, 256 x 5120 (5.4e9)
# 335 against 250 on the GPU, but twice the launches, and a layer of that size is bound by its host (617 us a step against
# 660); 2048 rows, 512 x 10240 (1.1e10) a layer step of 705 against 625; 8192 rows, 512 x 5 * 1024 (2.1e10) 1042 against 588.
MIN_WORK = 1 << 33

# Most rows and outputs: the kernel counts to the end of its last tile of 256 in 32 bits.
MAX_ROWS = (1 << 31) - 1 - 256


class Maxima(NamedTuple):
    """What the backward needs of the operands: bits of the largest magnitude of every column of the input, and of
    every column over all weights, in parts (None where no gradient asks for them)."""

    u_col: Optional[Tensor]
    w_col: Optional[Tensor]


def _matrix_ok(t: Tensor) -> bool:
    return (t.dtype is torch.float32 and t.is_cuda and t.dim() == 2 and t.stride(1) == 1 and t.stride(0) >= t.shape[1]
            and t.stride(0) % 4 == 0 and t.stride(0) < 1 << 20 and t.data_ptr() % 16 == 0)


def usable(u: Tensor, weights: Sequence[Tensor]) -> bool:
    """Whether u [.., K] times the transposes of the weights [N, K] may take the split products."""
    n, k = weights[0].shape
    if u.dtype is not torch.float32 or u.numel() * n * len(weights) < MIN_WORK:
        return False
    if not u.is_cuda or torch.is_autocast_enabled("cuda") or n % 4 or k % 4:
        return False
    if u.numel() // k > MAX_ROWS or n > MAX_ROWS:
        return False
    if not _matrix_ok(u.reshape(-1, k)):
        return False
    return all(_matrix_ok(w) and w.shape == (n, k) and w.stride(0) == weights[0].stride(0) and w.device == u.device
               for w in weights)


def forward(u: Tensor, weights: Sequence[Tensor], biases: Sequence[Optional[Tensor]], need_du: bool, need_dw: bool
            ) -> Tuple[List[Tensor], Maxima]:
    """u w^T + bias for every weight (call `usable` first), and the maxima a backward wants."""
    native = hip_scan._native or hip_scan._load_native()
    outs, u_col, w_col = native.split_forward(u, weights, biases, need_dw | need_du << 1)
    return outs, Maxima(u_col, w_col)


def backward(grads: Sequence[Tensor], u: Tensor, weights: Sequence[Tensor], saved: Maxima, need_du: bool, need_dw: bool
             ) -> Tuple[Optional[Tensor], List[Optional[Tensor]]]:
    """Gradients of the input (summed over the weights) and of every weight from the outputs' gradients [rows, N]."""
    native = hip_scan._native or hip_scan._load_native()
    du, dws = native.split_backward(grads, u, weights, saved.u_col, saved.w_col, need_du | need_dw << 1)
    return du, (dws if need_dw else [None] * len(weights))


__all__ = ["usable", "forward", "backward", "Maxima"]
