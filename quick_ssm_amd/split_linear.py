"""Linear maps of the SSM layer over fp32 parameters, on the bf16 matrix cores (csrc/gemm_split.hip).

A layer with fp32 parameters spends nine tenths of its time in its projections (quick_ssm/layers.py:76-80,106): the
library's fp32 products run at the fp32 MFMA rate, a sixteenth of the bf16 one.  `qssm_gemm_f32` takes every element as
the sum of three bf16 values, which hold all of its bits, and accumulates six products in fp32; measured against float64
it is 1.2 (rows of two nonzeros) to nine times (long sums) closer than fp32 products, and 2 % further off for a sum of one
nonzero pair (2.60e-8 against 2.54e-8).  Here is the rule for when it is used; scratch and the calls are in
csrc/torch_scan.cpp, the autograd functions that use them in quick_ssm_amd/layers.py.
"""
from __future__ import annotations

from typing import List, Optional, Sequence, Tuple

import torch

from . import hip_scan

Tensor = torch.Tensor

# Multiply-adds (over all weights of a launch) below which the library's product stays.  GPU us for output, input gradient
# and weight gradient, library against these: 2^30 (4096 rows, 1024 -> 256) 24, 25, 30 against 41, 33, 42; 2^32.3 (4096 rows,
# 256 -> 5120) 103, 95, 133 against 83, 66, 69; 2^33.3 (4096 rows, 512 -> 5120) 168, 154, 171 against 130, 113, 115.  They
# cross near 2^31; the line is above the copy task's stack (2^32.3 a layer), whose six layers in fp16 carry a difference in a
# product's last bits on to 3e-3 of a gradient: at that size outputs and input gradients stay the library's products.  (Weight
# gradients, on which nothing else in a step depends, are this package's from layers._GRADIENT_WORK on.)
MIN_WORK = 1 << 33

# An input narrower than this has few stages to fill a tile's pipeline with before its results are stored: 16384 rows,
# 64 -> 2560 would be two.  At 128 columns the library's 109 us stand against 97, at 208 -> 4160 357 against 244.
MIN_INFERENCE_WIDTH = 128

# Below 256 columns the outputs (of all weights) have to fill their tiles as well: 1572869 rows, 128 -> 128 546 against 587,
# 2139100 rows, 128 -> 32 338 against 558, 118843 rows, 144 -> 512 176 against 183; from 1024 outputs on 1.0 to 2.2 times the
# library's speed.
_NARROW, _NARROW_OUTPUTS = 256, 1024

# Most rows and outputs: the kernel counts to the end of its last tile of 128 in 32 bits.
MAX_ROWS = (1 << 31) - 1 - 128


def _matrix_ok(t: Tensor) -> bool:
    return (t.dtype is torch.float32 and t.is_cuda and t.dim() == 2 and t.stride(1) == 1 and t.stride(0) >= t.shape[1]
            and t.stride(0) % 4 == 0 and t.stride(0) < 1 << 20 and t.data_ptr() % 16 == 0)


def usable(u: Tensor, weights: Sequence[Tensor], gradients: bool = True) -> bool:
    """Whether u [.., K] times the transposes of the weights [N, K] may take the split products; `gradients`: theirs will
    be asked for."""
    n, k = weights[0].shape
    if u.dtype is not torch.float32 or u.numel() * n * len(weights) < MIN_WORK:
        return False
    if not u.is_cuda or torch.is_autocast_enabled("cuda") or n % 4 or k % 4:
        return False
    if u.numel() // k > MAX_ROWS or n > MAX_ROWS:
        return False
    if not gradients and (k < MIN_INFERENCE_WIDTH or (k < _NARROW and n * len(weights) < _NARROW_OUTPUTS)):
        return False
    if not _matrix_ok(u.reshape(-1, k)):
        return False
    return all(_matrix_ok(w) and w.shape == (n, k) and w.stride(0) == weights[0].stride(0) and w.device == u.device
               for w in weights)


def forward(u: Tensor, weights: Sequence[Tensor], biases: Sequence[Optional[Tensor]], need_du: bool = True,
            need_dw: bool = True) -> Tuple[List[Tensor], None]:
    """u w^T + bias for every weight (call `usable` first), and what a backward that asks for `need_du` and `need_dw`
    wants kept besides the operands: nothing, they are split where they are used."""
    native = hip_scan._native or hip_scan._load_native()
    return native.split_forward(u, weights, biases), None


def backward(grads: Sequence[Tensor], u: Tensor, weights: Sequence[Tensor], saved: None, need_du: bool, need_dw: bool
             ) -> Tuple[Optional[Tensor], List[Optional[Tensor]]]:
    """Gradients of the input (summed over the weights) and of every weight from the outputs' gradients [rows, N]."""
    native = hip_scan._native or hip_scan._load_native()
    du, dws = native.split_backward(grads, u, weights, need_du | need_dw << 1)
    return du, (dws if need_dw else [None] * len(weights))


__all__ = ["usable", "forward", "backward"]
