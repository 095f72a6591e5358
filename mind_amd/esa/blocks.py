"""The packed pre-norm blocks as one autograd function each.

``sab_block`` and ``pma_block`` run the computation of
``masked_layers._sab_separate`` / ``_pma_separate`` (the reference's
SABComplete.forward and PMAComplete.forward, esa/masked_layers.py:418-483,
574-621), but record one autograd node for a block instead of seven, and call
the kernels without the layers between: the norms and the attention are the
separate functions', a Linear runs with what follows it in one kernel, and so
do its input gradients, where linear.py says so.  A small batch's step is
bound by the host: a block's forward and backward issue about 35 launches,
and an autograd function around each costs more than the launch (64 small
molecules in fp32, three blocks, with the attention's dispatch, on the
separate functions' kernels: 3.48 -> 2.76 ms per train step).  The gradients
of a block's shared inputs are added inside its GEMMs and kernels, with at
most the roundings of the separate nodes.

They take the calls that nothing else has to see as single operations
(``eager.plain``), over the dtypes the kernels compute in: bf16 autocast with
fp32 parameters, or fp32 throughout.  Everything else stays with the separate
functions, which also serve a backward that is differentiated again.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch
from torch import nn

from . import attention
from .activations import Mish, mab_residual_backward, mish_backward
from .attention import HEAD_DIMS, attn_bwd, attn_fwd, pma_backward, pma_forward
from .eager import Unrecorded, call, plain
from .layer_norm import f32_values, ln_backward, ln_forward, supported
from .linear import (cast_param, hookless, input_grad, linear_outputs, linear_then_add, linear_then_mab,
                     linear_then_mish, on_boundary, weight_bias_grads)
from .mha import PMA
from .mlp_utils import SmallMLP


def _mlp_layers(blk) -> list[nn.Linear] | None:
    """The Linears of the block's MLP when it is Linear (-> Mish -> Linear)* without hooks, [] without an MLP, None
    for any other."""
    if not blk.use_mlp:
        return []
    glob = nn.modules.module
    if (type(blk.mlp) is not SmallMLP or "forward" in vars(blk.mlp) or not hookless(blk.mlp) or blk.mlp._backward_hooks
            or blk.mlp._backward_pre_hooks or glob._global_forward_hooks or glob._global_forward_pre_hooks
            or glob._global_backward_hooks or glob._global_backward_pre_hooks):
        return None
    layers = list(blk.mlp.mlp)
    for i, m in enumerate(layers):
        if type(m) not in ((nn.Linear,) if i % 2 == 0 else (Mish, nn.Mish)) or not hookless(m):
            return None
    return layers[::2] if len(layers) % 2 else None


def _compute_dtype(x: torch.Tensor, params):
    """The dtype the block's GEMMs run in: bf16 under bf16 autocast, fp32 where everything is fp32; None where the
    block is not taken."""
    if not x.is_cuda or x.dtype != torch.float32 or x.shape[0] == 0:
        return None
    if any(p is not None and (p.dtype != torch.float32 or p.device != x.device) for p in params):
        return None   # torch's own operations say what is wrong with a mixture
    if not torch.is_autocast_enabled("cuda"):
        return torch.float32
    return torch.bfloat16 if torch.get_autocast_dtype("cuda") == torch.bfloat16 else None


def _held(blk, mab) -> bool:
    """Whether the block's parameters are its modules' own: a subclass, as a parametrization makes it, may compute them
    with every look (and a spectral norm moves its estimate with it), where the separate functions look once."""
    return (all(type(fc) is nn.Linear for fc in (mab.fc_q, mab.fc_k, mab.fc_v, mab.fc_o))
            and all(type(n.ln) is nn.LayerNorm for n in (blk.norm, blk.norm_mlp)))


def _block_args(blk, mab, mlp):
    """The block's parameters in the functions' order."""
    args = [blk.norm.ln.weight, blk.norm.ln.bias]
    for fc in (mab.fc_q, mab.fc_k, mab.fc_v, mab.fc_o):
        args += (fc.weight, fc.bias)
    if mlp:
        args += (blk.norm_mlp.ln.weight, blk.norm_mlp.ln.bias)
    for fc in mlp:
        args += (fc.weight, fc.bias)
    return args


class _Setup:
    """What a block's function needs besides tensors."""

    def __init__(self, blk, tokens, mab, mlp, dt, dropout_p, again):
        self.eps = (blk.norm.ln.eps, blk.norm_mlp.ln.eps)
        self.heads, self.max_items, self.cu = mab.num_heads, tokens.max_items, tokens.cu_seqlens
        self.dt, self.amp, self.n_mlp = dt, dt != torch.float32, len(mlp)
        self.dropout = (dropout_p, attention.draw_dropout_seed() if dropout_p > 0.0 else 0)
        self.again = again   # (block, x, seed) -> the block's output through the separate functions
        self.mask = {}
        # whole stages of the fused products both ways, for the parameters themselves or (amp) their contiguous casts
        self.fused = all(fc.weight.dim() == 2 and fc.weight.is_contiguous() and max(fc.weight.shape) <= 16384
                         and fc.weight.shape[0] % 32 == 0 and fc.weight.shape[1] % 32 == 0
                         and (self.amp or all(t is None or (t.is_contiguous() and t.data_ptr() % 16 == 0)
                                              for t in (fc.weight, fc.bias)))
                         for fc in (mab.fc_q, mab.fc_k, mab.fc_v, mab.fc_o, *mlp))


def _fitting(d: int, mab, mlp) -> bool:
    """Whether the Linears' parameters have the shapes that the block's kernels read: D to D around the attention, a
    chain from D to D in the MLP (replaced or pruned parameters may not; F.linear checks them)."""
    sizes, last = [(fc, d, d) for fc in (mab.fc_q, mab.fc_k, mab.fc_v, mab.fc_o)], d
    for i, fc in enumerate(mlp):
        out = d if i + 1 == len(mlp) else fc.weight.shape[0]
        sizes.append((fc, out, last))
        last = out
    return all(fc.weight.shape == (o, i) and (fc.bias is None or fc.bias.shape == (o,)) for fc, o, i in sizes)


def _layer(cls, **attrs):
    """A module of type ``cls`` with these plain attributes and nothing registered."""
    m = cls.__new__(cls)
    nn.Module.__init__(m)
    m.__dict__.update(attrs)
    return m


def _stand_in(setup, d, params, seeds=None):
    """The block as its forward found it, for the separate functions: these parameters (``_block_args``' order), its
    dropout.  The module itself may hold others by now (functional calls) or be in another mode."""
    it = iter(params)

    def norm(eps):
        return SimpleNamespace(ln=_layer(nn.LayerNorm, weight=next(it), bias=next(it), normalized_shape=(d,), eps=eps))

    def linear():
        return _layer(nn.Linear, weight=next(it), bias=next(it))

    blk = SimpleNamespace(idx=1 if setup.mask else 0, use_mlp=setup.n_mlp > 0, residual_dropout=0.0,
                          norm=norm(setup.eps[0]))
    mab = SimpleNamespace(fc_q=linear(), fc_k=linear(), fc_v=linear(), fc_o=linear(), num_heads=setup.heads, dim_V=d,
                          dropout_p=setup.dropout[0], training=True)
    blk.sab = blk.pma = SimpleNamespace(mab=mab, S=seeds)
    if setup.n_mlp:
        blk.norm_mlp = norm(setup.eps[1])
        layers = [linear()]
        for _ in range(setup.n_mlp - 1):
            layers += (Mish(), linear())
        blk.mlp = _layer(SmallMLP, mlp=layers)
    return blk


def _versions(params, recorded: bool):
    """How often each parameter has been changed in place so far."""
    return [p._version for p in params if p is not None] if recorded else None


def _rebuilt(ctx, x, params, g, seeds=None):
    """The gradients of x, the seeds (where there are any) and the parameters by the separate functions, for a
    backward that is itself differentiated.  The parameters are not among the saved tensors: an ordinary backward
    takes the casts and statistics that the forward kept, so a bias, or under autocast a weight, may be changed in
    place before it."""
    setup, needs = ctx.setup, ctx.needs_input_grad[1:]
    if _versions(ctx.inputs, True) != ctx.versions:
        raise RuntimeError("one of the variables needed for gradient computation has been modified by an inplace "
                           "operation: a parameter of a packed block, whose backward is to be differentiated again")
    inputs = [x] + ([] if seeds is None else [seeds]) + list(params)
    with torch.enable_grad(), torch.autocast("cuda", setup.dt if setup.amp else None, enabled=setup.amp):
        out = setup.again(_stand_in(setup, x.shape[1], params, seeds), x, setup.dropout[1])
        got = iter(torch.autograd.grad(out, [t for t, n in zip(inputs, needs) if n], g, create_graph=True))
    return tuple(next(got) if n else None for n in needs)


def _norm(setup, x, w, b, eps, full):
    """(ln(x) in fp32 or None, the rows its Linear takes, statistics)."""
    if setup.amp:
        return ln_forward(x, f32_values(w), f32_values(b), eps, torch.float32, full, True)
    y, _, stats = ln_forward(x, f32_values(w), f32_values(b), eps, x.dtype, True, False)
    return y, y, stats


def _mlp_forward(x, params, residual, keep, fused):
    """Linear (-> Mish -> Linear)* plus the residual: (output, [the tensors _mlp_backward takes: a layer's input and
    weight and, before a Mish, z])."""
    saved = []
    for i in range(0, len(params), 2):
        w, b = cast_param(params[i], x.dtype), cast_param(params[i + 1], x.dtype)
        saved += (x, w)
        if i + 2 < len(params):
            z, x = linear_then_mish(x, w, b, keep, fused)
            saved.append(z)
    if residual.dtype == torch.float32:
        return linear_then_add(x, w, b, residual, fused), saved
    return linear_outputs(x, [(w, b)], fused)[0] + residual, saved


# Token counts up to which a block's weight gradients wait for the end of its backward and run in one launch: the
# launches of single weights leave the chip partly idle at their ends and each costs the host.  Six weights of a SAB
# block with an MLP, together / apart, us: fp32 128 wide (MLP 256) 92 / 136 at 33,000 tokens; bf16 256 (1024) 91 / 135
# at 33,000 and 145 / 203 at 65,000; 512 (2048) 230 / 304 at 33,000 and 457 / 491 at 65,000.  Up to the line every
# width gains.  Beyond, that is the width's matter: 512 loses from 100,000 tokens on (710 / 703; 131,000: 935 / 903),
# where a weight alone fills the chip, 192 (768) at 262,000 (482 / 456), while 256 and 128 gain still (131,000: 256 /
# 337, 92 / 143); and the operands of all six stay allocated to the end.
_TOGETHER = 65536


class _Grads:
    """The gradients of a block's inputs by position, those of its Linears from their (output gradient, input)."""

    def __init__(self, setup, needs, rows):
        self.needs, self.out, self.pairs = needs, [None] * len(needs), []
        self.together = setup.fused and rows <= _TOGETHER

    def add(self, *pairs):
        """(position of the weight, g, x), the bias one further; computed now unless they can wait."""
        self.pairs += pairs
        if not self.together:
            self.compute()

    def compute(self):
        by_rows = {}
        for pair in self.pairs:
            by_rows.setdefault(pair[1].shape[0], []).append(pair)
        for pairs in by_rows.values():
            got = weight_bias_grads([p[1:] for p in pairs], [self.needs[p[0]] for p in pairs],
                                    [self.needs[p[0] + 1] for p in pairs])
            for (i, _, _), pair in zip(pairs, got):
                self.out[i:i + 2] = pair
        self.pairs = []


def _mlp_backward(g, saved, grads, first, fused):
    """dx for the output gradient g in the compute dtype; the parameters from position ``first`` on go to ``grads``."""
    layers = [saved[i:i + 3] for i in range(0, len(saved), 3)]
    for i in range(len(layers) - 1, -1, -1):
        x, w = layers[i][:2]
        grads.add((first + 2 * i, g, x))
        g = input_grad([(g, w)], fused, mish_z=layers[i - 1][2] if i else None)
    return g


class _SabBlock(torch.autograd.Function):
    @staticmethod
    def forward(ctx, setup, x, *params):
        ln_w, ln_b, wq, bq, wk, bk, wv, bv, wo, bo = params[:10]
        t, d, h, keeps = x.shape[0], x.shape[1], setup.heads, not isinstance(ctx, Unrecorded)
        x1, xm, stats = _norm(setup, x, ln_w, ln_b, setup.eps[0], True)
        weights = [cast_param(p, setup.dt) for p in (wq, wk, wv, wo)]
        biases = [cast_param(p, setup.dt) for p in (bq, bk, bv, bo)]
        q, k, v = (y.view(t, h, d // h) for y in linear_outputs(xm, list(zip(weights[:3], biases[:3])), setup.fused))
        cu, n, (p, seed) = setup.cu, setup.max_items, setup.dropout
        o, lse = attn_fwd(q, k, v, cu, cu, n, n, 1.0 / math.sqrt(d // h), dropout_p=p, dropout_seed=seed, **setup.mask)
        z, x2 = linear_then_mab(o.view(t, d), weights[3], biases[3], x1, keeps, setup.fused)
        keep = [x, f32_values(ln_w), stats, xm, q, k, v, o, lse, z] + weights
        out = x2
        if setup.n_mlp:
            ln_w2, ln_b2 = params[10:12]
            _, ym, stats2 = _norm(setup, x2, ln_w2, ln_b2, setup.eps[1], False)
            out, saved = _mlp_forward(ym, params[12:], x2, keeps, setup.fused)
            keep += [x2, f32_values(ln_w2), stats2] + saved
        ctx.setup, ctx.n_keep, ctx.mask_keys = setup, len(keep), list(setup.mask)
        ctx.inputs, ctx.versions = params, _versions(params, keeps)
        ctx.save_for_backward(*keep, cu, *setup.mask.values())
        return out

    @staticmethod
    def backward(ctx, g):
        setup, needs, tensors = ctx.setup, ctx.needs_input_grad[1:], ctx.saved_tensors
        if torch.is_grad_enabled():
            return (None,) + _rebuilt(ctx, tensors[0], ctx.inputs, g)
        x, ln_w, stats, xm, q, k, v, o, lse, z, wq, wk, wv, wo = tensors[:14]
        cu, mask = tensors[ctx.n_keep], dict(zip(ctx.mask_keys, tensors[ctx.n_keep + 1:]))
        t, d = x.shape
        g, grads = on_boundary(g.contiguous()), _Grads(setup, needs, t)
        if setup.n_mlp:
            x2, ln_w2, stats2 = tensors[14:17]
            dy = _mlp_backward(g.to(setup.dt), tensors[17:ctx.n_keep], grads, 13, setup.fused)
            g, *grads.out[11:13] = ln_backward(x2, ln_w2, stats2, None if setup.amp else dy, dy if setup.amp else None,
                                               g, needs[11], needs[12])
        dz, g_o = mab_residual_backward(z, g)
        do = input_grad([(dz, wo)], setup.fused, g_o).view_as(o)
        grads.add((9, dz, o.view(t, d)))
        n, (p, seed) = setup.max_items, setup.dropout
        gq, gk, gv = (y.view(t, d) for y in attn_bwd(do, q, k, v, o, lse, cu, cu, n, n, 1.0 / math.sqrt(d // setup.heads),
                                                     dropout_p=p, dropout_seed=seed, **mask))
        # fp32: the norm's one output feeds the projections and the residual, whose gradient g starts the sum
        dxm = input_grad([(gq, wq), (gk, wk), (gv, wv)], setup.fused, None if setup.amp else g)
        grads.add((3, gq, xm), (5, gk, xm), (7, gv, xm))
        grads.compute()
        grads.out[:3] = ln_backward(x, ln_w, stats, g if setup.amp else dxm, dxm if setup.amp else None, None,
                                    needs[1], needs[2])
        return (None, *grads.out)


def sab_block(blk, x: torch.Tensor, tokens, masked: bool, attn_p: float, again) -> torch.Tensor | None:
    """The SABComplete block ``blk`` on packed tokens x [T, D], or None where this path does not take the call.
    ``again(blk, x, seed)`` computes a block through the separate functions."""
    mab, ln = blk.sab.mab, blk.norm.ln
    mlp = _mlp_layers(blk)
    if mlp is None or blk.residual_dropout > 0 or x.dim() != 2 or mab.dim_V != x.shape[1] or not _held(blk, mab):
        return None
    d, h = x.shape[1], mab.num_heads
    params = _block_args(blk, mab, mlp)
    dt = _compute_dtype(x, params)
    if (dt is None or d % h or d // h not in HEAD_DIMS or not supported(x, ln) or not supported(x, blk.norm_mlp.ln)
            or not _fitting(d, mab, mlp) or not plain(x, *params)):
        return None
    setup = _Setup(blk, tokens, mab, mlp, dt, attn_p, again)
    if masked:
        setup.mask = tokens.kernel_mask(padded=False)
    return call(_SabBlock, setup, x.contiguous(), *params)


class _PmaBlock(torch.autograd.Function):
    @staticmethod
    def forward(ctx, setup, x, seeds, *params):
        ln_w, ln_b, wq, bq, wk, bk, wv, bv, wo, bo = params[:10]
        (k_seeds, d), h, keeps = seeds.shape[1:], setup.heads, not isinstance(ctx, Unrecorded)
        _, xm, stats = _norm(setup, x, ln_w, ln_b, setup.eps[0], False)
        s = cast_param(seeds, setup.dt).reshape(k_seeds, d).contiguous()
        weights = [cast_param(p, setup.dt) for p in (wq, wk, wv, wo)]
        biases = [cast_param(p, setup.dt) for p in (bq, bk, bv, bo)]
        (q,) = linear_outputs(s, [(weights[0], biases[0])], setup.fused)
        k, v = linear_outputs(xm, list(zip(weights[1:3], biases[1:3])), setup.fused)
        q, k, v = (y.view(-1, h, d // h) for y in (q, k, v))
        o, lse = pma_forward(q, k, v, setup.cu, setup.max_items, 1.0 / math.sqrt(d // h), *setup.dropout)
        z, x2 = linear_then_mab(o.view(-1, d), weights[3], biases[3], None, keeps, setup.fused)
        keep = [x, f32_values(ln_w), stats, xm, s, q, k, v, o, lse, z] + weights
        out = x2
        if setup.n_mlp:
            ln_w2, ln_b2 = params[10:12]
            _, ym, stats2 = _norm(setup, x2, ln_w2, ln_b2, setup.eps[1], False)
            out, saved = _mlp_forward(ym, params[12:], x2, keeps, setup.fused)
            keep += [x2, f32_values(ln_w2), stats2] + saved
        ctx.setup, ctx.n_keep = setup, len(keep)
        ctx.inputs, ctx.versions = (seeds, *params), _versions((seeds, *params), keeps)
        ctx.save_for_backward(*keep, setup.cu)
        return out.view(-1, k_seeds, d)

    @staticmethod
    def backward(ctx, g):
        setup, needs, tensors = ctx.setup, ctx.needs_input_grad[1:], ctx.saved_tensors
        if torch.is_grad_enabled():
            return (None,) + _rebuilt(ctx, tensors[0], ctx.inputs[1:], g, ctx.inputs[0])
        x, ln_w, stats, xm, s, q, k, v, o, lse, z, wq, wk, wv, wo = tensors[:15]
        cu, seeds, d = tensors[ctx.n_keep], ctx.inputs[0], x.shape[1]
        g, grads = on_boundary(g.contiguous()).view(-1, d), _Grads(setup, needs, x.shape[0])
        if setup.n_mlp:
            x2, ln_w2, stats2 = tensors[15:18]
            dy = _mlp_backward(g, tensors[18:ctx.n_keep], grads, 14, setup.fused)
            g, *grads.out[12:14] = ln_backward(x2, ln_w2, stats2, None if setup.amp else dy, dy if setup.amp else None,
                                               g, needs[12], needs[13])
        dz = mish_backward(z, g)
        do = input_grad([(dz, wo)], setup.fused, g).view_as(o)
        grads.add((10, dz, o.view(-1, d)))
        gq, gk, gv = (y.view(-1, d) for y in pma_backward(do, q, k, v, o, lse, cu, setup.max_items,
                                                          1.0 / math.sqrt(d // setup.heads), *setup.dropout))
        if needs[1]:
            grads.out[1] = input_grad([(gq, wq)], setup.fused).view(seeds.shape).to(seeds.dtype)
        dxm = input_grad([(gk, wk), (gv, wv)], setup.fused)
        grads.add((4, gq, s), (6, gk, xm), (8, gv, xm))
        grads.compute()
        grads.out[0], *grads.out[2:4] = ln_backward(x, ln_w, stats, None if setup.amp else dxm,
                                                    dxm if setup.amp else None, None, needs[2], needs[3])
        return (None, *grads.out)


def pma_block(blk, x: torch.Tensor, tokens, attn_p: float, again) -> torch.Tensor | None:
    """The PMAComplete block ``blk`` over packed keys x [T, D] -> [B, k, D], or None where this path does not take
    the call (as ``sab_block``; a seed count equal to the sets' padded size has a residual of its own)."""
    mab, ln = blk.pma.mab, blk.norm.ln
    mlp = _mlp_layers(blk)
    if mlp is None or blk.residual_dropout > 0 or x.dim() != 2 or type(blk.pma) is not PMA or not _held(blk, mab):
        return None
    d, h, seeds = x.shape[1], mab.num_heads, blk.pma.S
    if mab.dim_V != d or seeds.shape[2] != d or seeds.shape[1] == tokens.max_items or tokens.batch_size < 1:
        return None
    params = _block_args(blk, mab, mlp)
    dt = _compute_dtype(x, [seeds] + params)
    if (dt is None or d % h or d // h not in HEAD_DIMS or not supported(x, ln) or not supported(x, blk.norm_mlp.ln)
            or not _fitting(d, mab, mlp) or not plain(x, seeds, *params)):
        return None
    return call(_PmaBlock, _Setup(blk, tokens, mab, mlp, dt, attn_p, again), x.contiguous(), seeds, *params)
