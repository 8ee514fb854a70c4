"""`SSM` and `RMSNorm`: the layer that feeds the scan.

Same constructor arguments, parameter names (so state dicts interchange) and forward keywords as
the reference's quick_ssm/layers.py:9-107.  The projections are torch GEMMs, except over fp32
parameters, where they are split products on the bf16 matrix cores (quick_ssm_amd/split_linear.py), and
except weight gradients over many rows (`_weight_gradient`); the gate
activations and casts between them and the scan happen inside the scan's own launches when the
projections are stored as the 16-bit compute dtype (quick_ssm_amd/gated_scan.py) and are one fused HIP
pass otherwise (quick_ssm_amd/gates.py),
the pre-norm is one fused HIP pass each way (quick_ssm_amd/norm.py), and the scan is the HIP path.  Roles of the projections
(quick_ssm/test_swiglu_equiv.py:60-70): A_proj -> forget gate a, B_proj -> the scan's input x,
D_proj -> input gate b, C_proj_a/C_proj_b -> SwiGLU output gate c, out_proj -> output.
"""
from __future__ import annotations

from typing import Optional

import torch
import torch.nn as nn

from . import _lib
from . import gated_scan as _gated
from . import hip_scan
from . import scan_interface as _scan_interface
from . import split_linear
from .gates import gate_prologue, gate_prologue_wide
from .norm import rms_norm
from .scan_interface import scan


class RMSNorm(nn.Module):
    """x * weight / sqrt(mean(x^2) + eps) over the last axis (quick_ssm/layers.py:9-17)."""

    def __init__(self, hidden_size: int, eps: float = 1e-5, dtype=torch.float32, device=None):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(hidden_size, dtype=dtype, device=device))

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return rms_norm(x, self.weight, self.eps)


_CODES = {torch.float32: _lib.QSSM_F32, torch.float16: _lib.QSSM_F16, torch.bfloat16: _lib.QSSM_BF16}
_COLSUM_PARTIAL_ROWS = 64


def column_sum(g2: torch.Tensor) -> torch.Tensor:
    """Sum over the rows of a [rows, S] matrix: the bias gradient of a linear map from its output's gradient.

    GPU matrices with unit column stride (a column block of a wider matrix is fine) take `qssm_colsum`: two small
    launches, a fixed summation order; a library reduction of this shape costs as much as the layer's scan at the
    copy task's size.  Everything else is `g2.sum(0)`."""
    rows, S = g2.shape
    if not (g2.is_cuda and g2.dtype in _CODES and S > 0 and rows > 0 and g2.stride(1) == 1 and g2.stride(0) >= S):
        return g2.sum(0)
    return (hip_scan._native or hip_scan._load_native()).column_sum(g2, _COLSUM_PARTIAL_ROWS)


# Rows, or multiply-adds in fp32, from which a weight gradient is this package's own product.  Its sums are as long as there
# are rows, and the library gives a tile of it to one workgroup, most of the GPU idle.  16 bits: the measured line is at
# qssm_weight_gradient_suits.  fp32, us for the library's product and for these (csrc/gemm_split.hip): 2^32.3 (4096 rows, 5120 x
# 256) 120 and 68, (1024 rows, 5120 x 1024) 88 and 74, (512 rows, 10240 x 1024) 86 and 84; 2^32 (4096 rows, 1024 x 1024) 63 and
# 67; with few rows a tile is all start and end and only memory counts: (128 rows, 8192 x 8192) 155 and 144, but (64 rows, 8192
# x 16384) 193 and 213, (16 rows, 40960 x 8192) 248 and 508; with many rows earlier: 8192 rows, 256 x 1024 55 and 46, 128 x 128
# 45 and 36, 16384 rows, 128 x 512 99 and 47 (and never below 20 columns, csrc/torch_scan.cpp).
# (No result of a step but the gradient itself depends on its last bits, as those of split_linear.MIN_WORK do.)
_GRADIENT_ROWS, _GRADIENT_WORK, _GRADIENT_FEW_ROWS = 8192, 1 << 32, 128


def _weight_gradient(g2: torch.Tensor, u2: torch.Tensor) -> torch.Tensor:
    """The gradient of a linear map's weight from its outputs' gradient and its inputs ([rows, N], [rows, K])."""
    rows, n = g2.shape
    if ((rows >= _GRADIENT_ROWS
         or (rows >= _GRADIENT_FEW_ROWS and g2.dtype is torch.float32 and rows * n * u2.shape[1] > _GRADIENT_WORK))
            and g2.is_cuda and not (torch.is_grad_enabled() or torch.is_autocast_enabled("cuda") or _scan_interface._followed_by_torch())):
        native = hip_scan._native or hip_scan._load_native()
        dw = native.weight_gradient(g2, u2)
        if dw is not None:
            return dw
    return g2.t() @ u2


def _products(ctx, u: torch.Tensor, weights, biases):
    """u w^T + bias for every weight as split products, inside an autograd function's forward."""
    u2 = u.reshape(-1, u.shape[-1])
    ctx.split = True
    outs, _ = split_linear.forward(u2, weights, biases, ctx.needs_input_grad[0], any(ctx.needs_input_grad[1:]))
    return [t.view(*u.shape[:-1], t.shape[-1]) for t in outs]


def _product(ctx, u: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    """One of them, as a split product where that applies, else torch's.  (Small layers are bound by the interpreter: a
    16-bit one gets no further than its type.)"""
    if (u.dtype is torch.float32 and u.numel() * weight.shape[0] >= split_linear.MIN_WORK
            and split_linear.usable(u, (weight,), any(ctx.needs_input_grad))):
        return _products(ctx, u, (weight,), (bias,))[0]
    ctx.split = False
    return torch.nn.functional.linear(u, weight, bias)


def _product_gradients(ctx, grads, u: torch.Tensor, weights, need_du: bool, need_dw: bool):
    """Gradients of the input and of the weights from the outputs' gradients ([rows, N] each).  A backward that is
    itself recorded (create_graph) takes torch's products, which autograd can follow."""
    u2 = u.reshape(-1, u.shape[-1])
    if ctx.split and not torch.is_grad_enabled():
        du, dws = split_linear.backward(grads, u2, weights, None, need_du, need_dw)
        return (None if du is None else du.view_as(u)), dws
    du = None
    if need_du:
        du = grads[0] @ weights[0]
        for g, w in zip(grads[1:], weights[1:]):
            du = du + g @ w
        du = du.view_as(u)
    return du, [g.t() @ u2 if need_dw else None for g in grads]


class _LinearBias(torch.autograd.Function):
    """u @ weight^T + bias, as `torch.nn.functional.linear`, with the bias gradient from `column_sum`."""

    @staticmethod
    def forward(ctx, u, weight, bias):
        ctx.save_for_backward(u, weight)
        return _product(ctx, u, weight, bias)

    @staticmethod
    def backward(ctx, g):
        u, weight = ctx.saved_tensors
        need = ctx.needs_input_grad
        g2 = g.reshape(-1, g.shape[-1])
        if ctx.split:
            du, (dw,) = _product_gradients(ctx, [g2], u, [weight], need[0], need[1])
        else:
            du = (g2 @ weight).view_as(u) if need[0] else None
            dw = _weight_gradient(g2, u.reshape(-1, u.shape[-1])) if need[1] else None
        db = column_sum(g2) if need[2] else None
        return du, dw, db


class _PackedProjection(torch.autograd.Function):
    """u -> u @ wide_w^T + wide_b, where wide_w [5 S, H] and wide_b [5 S] are the memory of the five projection
    weights and of A_proj's bias (`SSM._packed_parameters`).  The five weights and the bias are passed as well so
    that autograd routes their gradients: one GEMM gives the gradient of the wide weight, whose row blocks go to the
    five parameters; the bias gradient is summed over A_proj's block only."""

    @staticmethod
    def forward(ctx, u, w_a, w_b, w_ca, w_cb, w_d, bias_a, wide_w, wide_b):
        ctx.save_for_backward(u, wide_w)
        return _product(ctx, u, wide_w, wide_b)

    @staticmethod
    def backward(ctx, g):
        u, wide_w = ctx.saved_tensors
        need = ctx.needs_input_grad
        S = wide_w.shape[0] // 5
        g2 = g.reshape(-1, g.shape[-1])
        blocks = [None] * 5
        if ctx.split:
            du, (dw,) = _product_gradients(ctx, [g2], u, [wide_w], need[0], any(need[1:6]))
        else:
            du = (g2 @ wide_w).view_as(u) if need[0] else None
            dw = _weight_gradient(g2, u.reshape(-1, u.shape[-1])) if any(need[1:6]) else None   # [5 S, H]
        if dw is not None:
            blocks = [dw[k * S:(k + 1) * S] if need[1 + k] else None for k in range(5)]
        dbias = column_sum(g2[:, :S]) if need[6] else None
        return (du, *blocks, dbias, None, None)


def _bias_gradient(g2: torch.Tensor) -> torch.Tensor:
    """`column_sum`, or torch's sum where the backward is itself recorded."""
    return g2.sum(0) if torch.is_grad_enabled() else column_sum(g2)


class _WideProjections(torch.autograd.Function):
    """The five projections of a 16-bit layer in training as one product over their concatenated weights, [.., 5 S] out.

    What it is for is the backward: one product over 5 S k's for the input's gradient instead of five and four additions,
    and one for all weights, whose five [S, H] products alone leave most of the GPU idle (K is the number of rows).  Unlike
    `_PackedProjection` the parameters keep their own memory.  They are concatenated by either pass and the copy is not
    kept between the two (it would hold all projection weights of every layer a second time until the backward: 42 MB at
    hidden 1024, state 4096); each copy of that size takes 32 us.  Layer step, five products -> one, bf16, at 2^24 and 2^26
    elements per output: hidden 1024 state 4096 1002 -> 993 and 3164 -> 3049 us, 512 and 2048 928 -> 705 and 2896 -> 2086, 512
    and 1024 1222 -> 809 and 3411 -> 2414, 256 and 1024 1043 -> 664 and 2824 -> 2034, 2048 and 2048 1578 -> 1409 and 5394 ->
    5386, where the five are efficient by themselves (`SSM._WIDE_PRODUCT_LIMIT`)."""

    @staticmethod
    def forward(ctx, u, w_a, w_b, w_ca, w_cb, w_d, bias_a):
        weights = (w_a, w_b, w_ca, w_cb, w_d)
        S = w_a.shape[0]
        wide_w = torch.cat(weights)                                                   # [5 S, H]
        wide_b = torch.cat((bias_a, bias_a.new_zeros(4 * S)))
        ctx.save_for_backward(u, *weights)
        return torch.nn.functional.linear(u, wide_w, wide_b)

    @staticmethod
    def backward(ctx, g):
        u, *weights = ctx.saved_tensors
        need = ctx.needs_input_grad
        S = weights[0].shape[0]
        g2 = g.reshape(-1, 5 * S)
        du = (g2 @ torch.cat(weights)).view_as(u) if need[0] else None
        blocks = [None] * 5
        if any(need[1:6]):
            dw = _weight_gradient(g2, u.reshape(-1, u.shape[-1]))                     # [5 S, H]
            blocks = [dw[k * S:(k + 1) * S] if need[1 + k] else None for k in range(5)]
        return (du, *blocks, _bias_gradient(g2[:, :S]) if need[6] else None)


class _SplitProjections(torch.autograd.Function):
    """The five projections of a layer with fp32 parameters as one launch: the input's gradient is one product over 5 S
    k's instead of five products and four additions, and the five weight gradients are one launch."""

    @staticmethod
    def forward(ctx, u, w_a, w_b, w_ca, w_cb, w_d, bias_a):
        ctx.save_for_backward(u, w_a, w_b, w_ca, w_cb, w_d)
        return tuple(_products(ctx, u, [w_a, w_b, w_ca, w_cb, w_d], [bias_a, None, None, None, None]))

    @staticmethod
    def backward(ctx, *grads):
        u, *weights = ctx.saved_tensors
        need = ctx.needs_input_grad
        gs = [g.reshape(-1, g.shape[-1]) for g in grads]
        du, dws = _product_gradients(ctx, gs, u, weights, need[0], any(need[1:6]))
        dbias = _bias_gradient(gs[0]) if need[6] else None
        return (du, *(dw if need[1 + k] else None for k, dw in enumerate(dws)), dbias)


def _plain_linear(m: nn.Module) -> bool:
    """An `nn.Linear` whose call does nothing but the product: no hooks, no replaced class or forward."""
    return (type(m) is nn.Linear and "forward" not in m.__dict__ and type(m.weight) is nn.Parameter
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks))


class SSM(nn.Module):
    """Gated linear recurrence layer: norm -> five projections -> scan -> out projection (+ residual)."""

    def __init__(
        self,
        hidden_size: int,
        state_size_mult: float = 1.0,
        eps: float = 1e-5,
        dtype: torch.dtype = torch.float32,
        device: Optional[torch.device] = None,
        compute_dtype: torch.dtype = torch.float16,
        use_residual: bool = True,
        use_norm: bool = True,
    ):
        super().__init__()
        self.hidden_size = hidden_size
        self.state_size_dim = int(hidden_size * state_size_mult)
        self.compute_dtype = compute_dtype
        self.use_residual = use_residual
        self.use_norm = use_norm

        def proj(n_in: int, n_out: int, bias: bool) -> nn.Linear:
            return nn.Linear(n_in, n_out, bias=bias, device=device, dtype=dtype)

        # Creation order matches the reference so that seeded initialisation matches too.
        self.A_proj = proj(hidden_size, self.state_size_dim, True)
        self.B_proj = proj(hidden_size, self.state_size_dim, False)
        self.C_proj_a = proj(hidden_size, self.state_size_dim, False)
        self.C_proj_b = proj(hidden_size, self.state_size_dim, False)
        self.D_proj = proj(hidden_size, self.state_size_dim, False)
        self.out_proj = proj(self.state_size_dim, hidden_size, True)
        self.pre_norm = RMSNorm(hidden_size, eps=eps, dtype=dtype, device=device) if use_norm else nn.Identity()

    # Below this many elements per projection output a layer's step is bound by launches, not by their work.
    _BATCHED_PROJECTION_LIMIT = 1 << 23

    # Up to this many, a 16-bit layer in training still takes one product for the five projections (`_WideProjections`).
    _WIDE_PRODUCT_LIMIT = 1 << 26

    def _packed_parameters(self):
        """The five projection weights as one [5 S, H] tensor and a [5 S] bias (A_proj's, then zeros) that ARE the
        parameters' memory: each `nn.Linear.weight` is a row block of the wide tensor, `A_proj.bias` the head of the
        wide bias.  Parameter objects, names and values stay what they were (state dicts and optimizers see no
        difference); only where their data lives changes, once.  Whatever gives the parameters storage of their own
        again (`.to()`, `.half()`, loading into fresh tensors) is noticed here by their addresses and packed again."""
        ws = (self.A_proj.weight, self.B_proj.weight, self.C_proj_a.weight, self.C_proj_b.weight, self.D_proj.weight)
        S, H = self.state_size_dim, self.hidden_size
        packed = self.__dict__.get("_packed")
        if packed is not None:
            wide_w, wide_b = packed
            base, step = wide_w.data_ptr(), S * H * wide_w.element_size()
            if (wide_w.dtype == ws[0].dtype and wide_b.dtype == self.A_proj.bias.dtype
                    and all(w.data_ptr() == base + k * step for k, w in enumerate(ws))
                    and self.A_proj.bias.data_ptr() == wide_b.data_ptr()):
                return wide_w, wide_b
        with torch.no_grad():
            wide_w = torch.cat([w.data for w in ws])                              # [5 S, H]
            for k, w in enumerate(ws):
                w.data = wide_w[k * S:(k + 1) * S]
            bias = self.A_proj.bias
            wide_b = torch.cat((bias.data, bias.data.new_zeros(4 * S)))
            bias.data = wide_b[:S]
        self.__dict__["_packed"] = (wide_w, wide_b)
        return wide_w, wide_b

    def _wide_projection(self, u: torch.Tensor) -> Optional[torch.Tensor]:
        """All five projection outputs as one [.., 5 S] tensor (blocks in A, B, C_a, C_b, D order) from a single GEMM
        over the packed weights, for small layers; None for the others.

        The copy task's 12 x hidden 256 stack spends a training step on about a thousand launches of a few
        microseconds each: one GEMM forward and two backward per layer instead of five and ten cut both the host's
        and the GPU's time (the wide tensor's blocks are read in place by the gate kernels, and their gradients are
        written as blocks of one wide gradient).  The weights are not concatenated per call: the five parameters
        live in one tensor (`_packed_parameters`), and the gradient of that tensor is handed back as five row blocks.
        Large layers keep the separate GEMMs: theirs are efficient already."""
        S, H = self.state_size_dim, self.hidden_size
        rows = u.numel() // H
        if not (u.is_cuda and 0 < rows * S <= self._BATCHED_PROJECTION_LIMIT):
            return None
        wide_w, wide_b = self._packed_parameters()
        return _PackedProjection.apply(u, self.A_proj.weight, self.B_proj.weight, self.C_proj_a.weight,
                                       self.C_proj_b.weight, self.D_proj.weight, self.A_proj.bias, wide_w, wide_b)

    def _projections(self, look: bool):
        """The five projections in A, B, C_a, C_b, D order, and, if asked to look, whether their calls are nothing but
        products."""
        mods = (self.A_proj, self.B_proj, self.C_proj_a, self.C_proj_b, self.D_proj)
        plain = (look and all(_plain_linear(m) for m in mods) and not nn.modules.module._has_any_global_hook()
                 and self.A_proj.bias is not None and all(m.bias is None for m in mods[1:]))
        return mods, plain

    def _large_projections(self, u: torch.Tensor):
        """The projection outputs of a layer above `_BATCHED_PROJECTION_LIMIT`: one [.., 5 S] tensor for a 16-bit layer in
        training, or None and the five tensors (blocks in A, B, C_a, C_b, D order)."""
        half = u.dtype in (torch.float16, torch.bfloat16)
        grad = torch.is_grad_enabled()
        mods, plain = self._projections(grad or not half)
        if plain and u.is_cuda:
            weights, bias = [m.weight for m in mods], self.A_proj.bias
            if split_linear.usable(u, weights, grad):
                return None, _SplitProjections.apply(u, *weights, bias)
            if (half and grad and all(t.dtype == u.dtype for t in (*weights, bias))
                    and 0 < u.numel() // self.hidden_size * self.state_size_dim <= self._WIDE_PRODUCT_LIMIT
                    and not torch.is_autocast_enabled("cuda")
                    and (u.requires_grad or any(t.requires_grad for t in (*weights, bias)))):
                return _WideProjections.apply(u, *weights, bias), None
        return None, tuple(m(u) for m in mods)

    def gates(self, u: torch.Tensor):
        """The scan's four operands (x, a, b, c) from the normalised input, in `compute_dtype`."""
        forget, drive, out_gate, in_gate = gate_prologue(
            self.A_proj(u), self.B_proj(u), self.C_proj_a(u), self.C_proj_b(u), self.D_proj(u), self.compute_dtype)
        return drive, forget, in_gate, out_gate

    def forward(
        self,
        x: torch.Tensor,
        *,
        block_l: int = 256,
        checkpoint: bool = True,
        tile_b: Optional[int] = None,
        tile_d: Optional[int] = None,
        backend: str = "auto",
        scan_out_dtype: Optional[torch.dtype] = None,
    ) -> torch.Tensor:
        if (x.is_cuda and torch.cuda.is_current_stream_capturing() and torch.is_grad_enabled()
                and (x.requires_grad or any(p.requires_grad for p in self.parameters()))):
            # a recorded training step would also record the backward of the projections' bias and weight gradients
            # (library reductions with memset nodes), which does not replay reliably on this platform
            raise RuntimeError(
                "quick_ssm_amd.SSM: recording a differentiable forward into a HIP graph is not supported (the backward's "
                "torch library calls record memset nodes that do not replay reliably on this platform); record under "
                "torch.no_grad(), or run the training step eagerly.")
        skip = x if self.use_residual else 0
        u = self.pre_norm(x) if self.use_norm else x
        w_dtype = self.out_proj.weight.dtype
        out_dtype = w_dtype if scan_out_dtype is None else scan_out_dtype
        if backend in ("auto", "hip", "triton") and u.is_cuda and not _scan_interface._HONOR_TILES:
            # 16-bit projections stored as the compute dtype, or fp32 projections with fp32 y: the activations (and the
            # casts to the compute dtype) happen inside the scan's launches
            wide = self._wide_projection(u)
            if wide is None:
                wide, pre = self._large_projections(u)
            if wide is not None and _gated.supported_wide(wide, self.compute_dtype, out_dtype, checkpoint):
                y = _gated.gated_scan_wide(wide, out_dtype=out_dtype, compute_dtype=self.compute_dtype)
            elif wide is None and _gated.supported(pre, self.compute_dtype, out_dtype, checkpoint):
                y = _gated.gated_scan(*pre, out_dtype=out_dtype, compute_dtype=self.compute_dtype)
            else:
                if wide is not None:
                    forget, drive, out_gate, in_gate = gate_prologue_wide(wide, self.compute_dtype)
                else:
                    forget, drive, out_gate, in_gate = gate_prologue(*pre, self.compute_dtype)
                y = scan(x=drive, a=forget, b=in_gate, c=out_gate, block_l=block_l, checkpoint=checkpoint,
                         tile_b=tile_b, tile_d=tile_d, out_dtype=out_dtype, backend=backend)
            y = y if y.dtype == w_dtype else y.to(w_dtype)
            return _LinearBias.apply(y, self.out_proj.weight, self.out_proj.bias) + skip
        drive, forget, in_gate, out_gate = self.gates(u)
        y = scan(
            x=drive, a=forget, b=in_gate, c=out_gate,
            block_l=block_l, checkpoint=checkpoint, tile_b=tile_b, tile_d=tile_d,
            out_dtype=out_dtype,
            backend=backend,
        )
        return self.out_proj(y.to(w_dtype)) + skip


__all__ = ["SSM", "RMSNorm"]
