"""Mish and the MAB's ``out + mish(fc_o(out))`` epilogue on the gfx950 kernels.

``mab_epilogue(o, fc_o, residual)`` fuses the whole epilogue of a MAB on
packed rows: fc_o's GEMM, Mish and the residual(s) in one pass
(``esa_mish_fwd``, or ``esa_mab_residual_fwd`` with the block's fp32
residual stream), and a backward whose input gradient needs no add kernel.

``mish(z, residual)`` computes ``residual + mish(z)`` (``mish(z)`` without a
residual) in one pass, evaluated in fp32 and rounded once, through
``esa_mish_fwd``; its backward is ``esa_mish_bwd``.  It serves the reference's
``out = out + F.mish(self.fc_o(out))`` (esa/mha.py:87,
esa/mha_flash_varlen.py:120,195), the MLP activations ``nn.Mish()``
(esa/mlp_utils.py:24-37) and the decoder head ``F.mish(decoder_linear(.))``
(esa/masked_layers.py:929,934).

Device tensors always go to the HIP kernels (an unbuilt library raises); CPU
tensors, which the kernels cannot take, use ``torch.nn.functional.mish``.
"""
from __future__ import annotations

import torch
from torch import nn
from torch.nn import functional as F

from .. import _lib
from .eager import call

_DTYPES = {torch.float32: _lib.ESA_F32, torch.bfloat16: _lib.ESA_BF16}


def mish_forward(z, residual=None):
    """esa_mish_fwd: residual + mish(z) of contiguous tensors of one dtype (mish(z) without a residual)."""
    y = torch.empty_like(z)
    _lib.check(_lib.load().esa_mish_fwd(z.data_ptr(), _lib.ptr(residual), z.numel(), _DTYPES[z.dtype], y.data_ptr(),
                                        _lib.stream_of(z)), "esa_mish_fwd")
    return y


def mish_backward(z, g):
    """esa_mish_bwd: g mish'(z), contiguous tensors of one dtype."""
    dz = torch.empty_like(z)
    _lib.check(_lib.load().esa_mish_bwd(z.data_ptr(), g.data_ptr(), z.numel(), _DTYPES[z.dtype], dz.data_ptr(),
                                        _lib.stream_of(z)), "esa_mish_bwd")
    return dz


def mab_residual_forward(z, o, x):
    """esa_mab_residual_fwd: x + r(o + mish(z)), x and the result fp32, r() the rounding to o's dtype."""
    y = torch.empty(x.shape, dtype=torch.float32, device=x.device)
    _lib.check(_lib.load().esa_mab_residual_fwd(z.data_ptr(), o.data_ptr(), x.data_ptr(), z.numel(), _DTYPES[o.dtype],
                                                y.data_ptr(), _lib.stream_of(o)), "esa_mab_residual_fwd")
    return y


def mab_residual_backward(z, g):
    """esa_mab_residual_bwd: (g mish'(z), r(g)) of the fp32 gradient g, in z's dtype."""
    dz, g_o = torch.empty_like(z), torch.empty_like(z)
    _lib.check(_lib.load().esa_mab_residual_bwd(z.data_ptr(), g.data_ptr(), z.numel(), _DTYPES[z.dtype], dz.data_ptr(),
                                                g_o.data_ptr(), _lib.stream_of(z)), "esa_mab_residual_bwd")
    return dz, g_o


class _Mish(torch.autograd.Function):
    @staticmethod
    def forward(ctx, z, residual):
        z = z.contiguous()
        ctx.save_for_backward(z)
        ctx.has_residual = residual is not None
        return mish_forward(z, None if residual is None else residual.contiguous())

    @staticmethod
    def backward(ctx, g):
        (z,) = ctx.saved_tensors
        g = g.to(z.dtype).contiguous()
        return mish_backward(z, g), (g if ctx.has_residual else None)


def mish(z: torch.Tensor, residual: torch.Tensor | None = None) -> torch.Tensor:
    """``residual + mish(z)``, or ``mish(z)`` when residual is None."""
    if not z.is_cuda:
        return F.mish(z) if residual is None else residual + F.mish(z)
    if z.dtype not in _DTYPES:
        raise TypeError(f"mish: unsupported dtype {z.dtype}; use float32 or bfloat16")
    if residual is not None and (residual.dtype != z.dtype or residual.shape != z.shape):
        # Mixed precision or broadcasting: torch's promotion rules for the add.
        return residual + call(_Mish, z, None)
    return call(_Mish, z, residual)


class _MabEpilogue(torch.autograd.Function):
    """y = o + mish(fc_o(o)) (x is None) or y = x + r(o + mish(fc_o(o))) (x the block's fp32 residual, r() the
    rounding to o's dtype): fc_o's GEMM, then esa_mish_fwd / esa_mab_residual_fwd.  Backward: one kernel gives
    dz (and o's residual gradient r(g) when x is given), and o's gradient is r(g) + dz W in one GEMM (addmm,
    beta = 1)."""

    @staticmethod
    def forward(ctx, o, weight, bias, x):
        from .linear import cast_param, linear_fwd   # deferred: linear.py is a sibling with its own imports
        ctx.dtypes = (weight.dtype, None if bias is None else bias.dtype)   # the gradients are returned in these
        weight, bias = cast_param(weight, o.dtype), cast_param(bias, o.dtype)
        (z,) = linear_fwd(o, [(weight, bias)])
        y = mish_forward(z, o) if x is None else mab_residual_forward(z, o, x)
        ctx.save_for_backward(o, weight, z)
        ctx.has_x = x is not None
        return y

    @staticmethod
    def backward(ctx, g):
        from .linear import weight_bias_grads   # deferred: linear.py is a sibling with its own imports
        o, weight, z = ctx.saved_tensors
        if ctx.has_x:
            g = g.float().contiguous()
            dz, g_o = mab_residual_backward(z, g)
        else:
            g_o = g.to(z.dtype).contiguous()
            dz = mish_backward(z, g_o)
        wdt, bdt = ctx.dtypes
        do = torch.addmm(g_o, dz, weight) if ctx.needs_input_grad[0] else None
        ((dw, db),) = weight_bias_grads([(dz, o)], [ctx.needs_input_grad[1]],
                                        [bdt is not None and ctx.needs_input_grad[2]])
        return do, None if dw is None else dw.to(wdt), None if db is None else db.to(bdt), (g if ctx.has_x and ctx.needs_input_grad[3] else None)


def mab_epilogue(o: torch.Tensor, fc_o: nn.Linear, residual: torch.Tensor | None = None) -> torch.Tensor:
    """``o + mish(fc_o(o))`` (esa/mha.py:87) on 2-D token rows, plus the block residual when given
    (``residual + (o + mish(fc_o(o)))``, esa/masked_layers.py:471-472), fused on device tensors."""
    if not o.is_cuda:
        y = o + F.mish(fc_o(o))
        return y if residual is None else residual + y
    from .linear import compute_dtype
    w, b = fc_o.weight, fc_o.bias
    dt = compute_dtype(o, w, b)
    if dt not in _DTYPES or o.dim() != 2:
        o = o if dt is None else o.to(dt)
        y = mish(F.linear(o, w if dt is None else w.to(dt), b if dt is None or b is None else b.to(dt)), o)
        return y if residual is None else residual + y
    o = o.to(dt).contiguous()
    if residual is not None and (residual.dtype != torch.float32 or residual.shape != o.shape):
        return residual + call(_MabEpilogue, o, w, b, None)
    return call(_MabEpilogue, o, w, b, None if residual is None else residual.contiguous())


class _LinearMish(torch.autograd.Function):
    """y = mish(x W^T + b), an MLP's Linear -> Mish (esa/mlp_utils.py:18-37).  Forward: the GEMM, then
    esa_mish_fwd.  Backward: esa_mish_bwd writes dz; dx = dz W and the weight and bias gradients (one kernel,
    weight_bias_grads) follow.  Parameters enter in their own dtype and are cast
    inside, so their gradients are returned in it (fp32 under autocast)."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        from .linear import cast_param, linear_fwd   # deferred: linear.py is a sibling with its own imports
        ctx.dtypes = (weight.dtype, None if bias is None else bias.dtype)
        w, b = cast_param(weight, x.dtype), cast_param(bias, x.dtype)
        (z,) = linear_fwd(x, [(w, b)])
        ctx.save_for_backward(x, w, z)
        return mish_forward(z)

    @staticmethod
    def backward(ctx, g):
        from .linear import weight_bias_grads   # deferred: linear.py is a sibling with its own imports
        x, w, z = ctx.saved_tensors
        wdt, bdt = ctx.dtypes
        g = g.to(z.dtype).contiguous()
        dz = mish_backward(z, g)
        dx = dz.mm(w) if ctx.needs_input_grad[0] else None
        ((dw, db),) = weight_bias_grads([(dz, x)], [ctx.needs_input_grad[1]],
                                        [bdt is not None and ctx.needs_input_grad[2]])
        return dx, None if dw is None else dw.to(wdt), None if db is None else db.to(bdt)


def linear_mish(x: torch.Tensor, layer: nn.Linear) -> torch.Tensor:
    """``mish(layer(x))`` with the fused backward of _LinearMish on device tensors."""
    if not x.is_cuda:
        return F.mish(layer(x))
    from .linear import compute_dtype, linear
    dt = compute_dtype(x, layer.weight, layer.bias)
    if dt not in _DTYPES:
        return mish(linear(x, layer.weight, layer.bias))
    x = x.to(dt)
    lead = x.shape[:-1]
    y = call(_LinearMish, x.reshape(-1, x.shape[-1]).contiguous(), layer.weight, layer.bias)
    return y.view(*lead, layer.weight.shape[0])


class Mish(nn.Mish):
    """nn.Mish on the HIP kernel (no parameters; state dicts are unchanged)."""

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return mish(x)
