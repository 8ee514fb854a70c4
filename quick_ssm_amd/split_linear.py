"""Linear maps of the SSM layer over fp32 parameters, on the 16-bit matrix cores (csrc/gemm_split.hip).

A layer with fp32 parameters spends nine tenths of its time in its projections (quick_ssm/layers.py:76-80,106): the
library's fp32 products run at the fp32 MFMA rate, a sixteenth of the fp16 one.  `qssm_split_gemm` takes every element
as the sum of two scaled fp16 values and accumulates three products in fp32, with an error at or below that of fp32
products.  Here are the host side of it (maxima, scratch, the calls) and the three products of a linear map; the
autograd functions that use them are in quick_ssm_amd/layers.py.
"""
from __future__ import annotations

import ctypes
from typing import List, NamedTuple, Optional, Sequence, Tuple

import torch

from . import _lib

Tensor = torch.Tensor

# Multiply-adds below which the library's product stays, because the launches for the maxima cost more than is gained:
# 4096 rows, 256 x 5120 (5.4e9) takes 104 us against 97 forward, 8192 rows, 512 x 5 * 1024 (2.1e10) 214 against 334.
MIN_WORK = 1 << 33


class Maxima(NamedTuple):
    """What the backward needs of the operands: bits of the largest magnitude of every column of the input, and of
    every input column over all weights (None where no gradient asks for them)."""

    u_col: Optional[Tensor]
    w_col: Optional[Tensor]


def _matrix_ok(t: Tensor) -> bool:
    return (t.dtype is torch.float32 and t.is_cuda and t.dim() == 2 and t.stride(1) == 1 and t.stride(0) >= t.shape[1]
            and t.stride(0) % 4 == 0 and t.stride(0) < 1 << 20 and t.data_ptr() % 16 == 0)


def usable(u: Tensor, weights: Sequence[Tensor]) -> bool:
    """Whether u [rows, K] times the transposes of the weights [N, K] may take the split products."""
    if u.dtype is not torch.float32 or not u.is_cuda or torch.is_autocast_enabled("cuda"):
        return False
    n, k = weights[0].shape
    rows = u.shape[0]
    if n % 4 or k % 4 or rows * n * k * len(weights) < MIN_WORK or rows >= 1 << 31 or not _matrix_ok(u):
        return False
    return all(_matrix_ok(w) and w.shape == (n, k) and w.stride(0) == weights[0].stride(0) and w.device == u.device
               for w in weights)


def _maxima(mats: Sequence[Tensor], rows: str, cols: str) -> Tuple[List[Optional[Tensor]], List[Optional[Tensor]]]:
    """Bits of the largest magnitudes of the rows and columns of matrices of one shape: "each" matrix its own, one
    for all of them "joint"ly, or "none"."""
    n, (r, c) = len(mats), mats[0].shape
    n_row, n_col = ({"none": 0, "joint": 1, "each": n}[w] for w in (rows, cols))
    words = torch.zeros(n_row * r + n_col * c, dtype=torch.int32, device=mats[0].device)
    row = [words[k * r:(k + 1) * r] for k in range(n_row)]
    col = [words[n_row * r + k * c:n_row * r + (k + 1) * c] for k in range(n_col)]
    call = _lib.SplitAmaxCall(rows=r, ld=mats[0].stride(0), cols=c, count=n)
    for k, m in enumerate(mats):
        call.x[k] = m.data_ptr()
        if n_row:
            call.row[k] = row[k % n_row].data_ptr()
        if n_col:
            call.col[k] = col[k % n_col].data_ptr()
    with _lib.launch_stream(words.device) as stream:
        _lib.check(_lib.load().qssm_split_amax(ctypes.byref(call), stream))
    return row, col


def _product(a: Sequence[Tensor], b: Sequence[Tensor], out: Sequence[Tensor], amax_a: Sequence[Tensor],
             amax_b: Sequence[Tensor], K: int, a_kstrided: bool, b_kstrided: bool,
             bias: Sequence[Optional[Tensor]] = ()) -> None:
    """out[i] = a[i] b[i]^T (+ bias[i]), or out[0] = the sum of them all when there is one out for several pairs."""
    M, N = out[0].shape
    batch = len(out)
    segments = len(a) if batch == 1 else 1
    lib = _lib.load()
    splits = lib.qssm_split_gemm_splits(M, N, K, batch, segments)
    call = _lib.SplitGemmCall(lda=a[0].stride(0), ldb=b[0].stride(0), ldc=out[0].stride(0), M=M, N=N, K=K, batch=batch,
                              segments=segments, splits=splits, a_kstrided=a_kstrided, b_kstrided=b_kstrided)
    for k, (x, y) in enumerate(zip(a, b)):
        call.a[k], call.b[k] = x.data_ptr(), y.data_ptr()
    for k, t in enumerate(out):
        call.c[k], call.amax_a[k], call.amax_b[k] = t.data_ptr(), amax_a[k].data_ptr(), amax_b[k].data_ptr()
    for k, t in enumerate(bias):
        call.bias[k] = None if t is None else t.data_ptr()
    if splits > 1:
        partial = torch.empty(splits * batch * M * N, dtype=torch.float32, device=out[0].device)
        call.partial, call.partial_floats = partial.data_ptr(), partial.numel()
    with _lib.launch_stream(out[0].device) as stream:
        _lib.check(lib.qssm_split_gemm(ctypes.byref(call), stream))


def forward(u: Tensor, weights: Sequence[Tensor], biases: Sequence[Optional[Tensor]], need_du: bool, need_dw: bool
            ) -> Tuple[List[Tensor], Maxima]:
    """u w^T + bias for every weight (call `usable` first), and the maxima a backward wants."""
    rows = u.shape[0]
    n, k = weights[0].shape
    u_row, u_col = _maxima([u], "each", "each" if need_dw else "none")
    w_row, w_col = _maxima(weights, "each", "joint" if need_du else "none")
    outs = [torch.empty((rows, n), dtype=torch.float32, device=u.device) for _ in weights]
    biases = [None if t is None else t.contiguous() for t in biases]
    _product([u] * len(weights), weights, outs, u_row * len(weights), w_row, k, False, False, biases)
    return outs, Maxima(u_col[0] if u_col else None, w_col[0] if w_col else None)


def backward(grads: Sequence[Tensor], u: Tensor, weights: Sequence[Tensor], saved: Maxima, need_du: bool, need_dw: bool
             ) -> Tuple[Optional[Tensor], List[Optional[Tensor]]]:
    """Gradients of the input (summed over the weights) and of every weight from the outputs' gradients [rows, N]."""
    rows = u.shape[0]
    n, k = weights[0].shape
    gs = [g if _matrix_ok(g) and g.stride(0) == grads[0].stride(0) else None for g in grads]
    if any(g is None for g in gs):
        gs = [torch.empty((rows, n), dtype=torch.float32, device=u.device).copy_(g) for g in grads]
    g_row, g_col = _maxima(gs, "joint" if need_du else "none", "each" if need_dw else "none")
    du, dws = None, [None] * len(weights)
    if need_du:
        du = torch.empty((rows, k), dtype=torch.float32, device=u.device)
        _product(gs, weights, [du], g_row, [saved.w_col], n, False, True)
    if need_dw:
        dws = [torch.empty((n, k), dtype=torch.float32, device=u.device) for _ in weights]
        _product(gs, [u] * len(weights), dws, g_col, [saved.u_col] * len(weights), rows, True, True)
    return du, dws


__all__ = ["usable", "forward", "backward", "Maxima"]
