"""nn.Linear for the packed ESA blocks, with weight and bias gradients of their own.

On packed edge tokens a Linear's weight gradient dW = g^T x reduces over all
T tokens of the batch (T = 131,072 in the encoder-stack benchmark) into a
small [out, in] matrix: one GEMM with K = T has only a few dozen output tiles
for 256 CUs.  ``weight_bias_grads`` cuts it over the tokens in one kernel that
also sums the bias gradient's columns (esa_weight_grad: two launches for up to
eight Linears that share their rows), in fp32 and rounded to the weight's
dtype once, as the single GEMM's fp32 accumulator is.  Shapes and dtypes
outside the kernel's run as S batched GEMMs over token chunks (``weight_grad``)
and a column sum.  The packed blocks' forwards and input gradients run with
what follows them in esa_linear_fwd / esa_linear_dx where those are faster;
the autograd functions here keep F.linear and dx = g W.
Under autocast the inputs are cast as autocast casts F.linear's (x, weight
and bias to the autocast dtype); the autograd functions take the parameters
in their own dtype and cast them inside, so the fp32 weight and bias
gradients are returned as they are computed, in fp32, instead of being
rounded to the autocast dtype and cast back by a second kernel.

Reference: the nn.Linear layers of the MAB (esa/mha.py:12-15) and of the MLPs
(esa/mlp_utils.py:18-37).
"""
from __future__ import annotations

import contextlib
import contextvars
import ctypes

import torch
from torch import nn
from torch.nn import functional as F

from .. import _lib
from .eager import call

_MIN_CHUNK = 4096               # tokens per chunk: below, a chunk's GEMM is too short to pay
_MAX_PARTIAL = 16 * 1024 * 1024  # fp32 values of all partials (64 MiB)
_MAX_SPLIT = 32


def split_count(tokens: int, out_features: int, in_features: int) -> int:
    """Chunks S of the split-K weight gradient (1 = a single GEMM): the largest power of two <= 32 with chunks
    of >= 4096 tokens and S * out * in fp32 partials within 64 MiB."""
    s = 1
    while (2 * s <= _MAX_SPLIT and tokens // (2 * s) >= _MIN_CHUNK
           and 2 * s * out_features * in_features <= _MAX_PARTIAL):
        s *= 2
    return s


def weight_grad(g: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """g^T x for g [T, out], x [T, in] (same dtype) in fp32, by split_count(T, out, in) token chunks: the shapes
    and dtypes that esa_weight_grad does not take."""
    t, o = g.shape
    i = x.shape[1]
    s = split_count(t, o, i)
    # bf16 device operands: products accumulated and returned in fp32 by the GEMM itself (out_dtype), no casts
    kw = {} if g.dtype == torch.float32 or not g.is_cuda else {"out_dtype": torch.float32}
    if t < _MIN_CHUNK:
        return torch.mm(g.t(), x, **kw) if kw else g.t().float().mm(x.float())
    c = t // s
    t0 = s * c
    parts = torch.bmm(g[:t0].view(s, c, o).transpose(1, 2), x[:t0].view(s, c, i), **kw)
    dw = parts.sum(0)
    if t0 < t:   # fewer than S leftover tokens: added by the GEMM's epilogue
        dw = torch.addmm(dw, g[t0:].t(), x[t0:], **kw)
    return dw


_CODES = {torch.float32: _lib.ESA_F32, torch.bfloat16: _lib.ESA_BF16}


def _aligned(t: torch.Tensor) -> bool:
    return t.data_ptr() % 16 == 0


def on_boundary(t: torch.Tensor) -> torch.Tensor:
    """The contiguous t, or its copy where its memory starts off the 16-byte boundary that the kernels ask for."""
    return t if _aligned(t) else t.clone()


def column_sum(g: torch.Tensor) -> torch.Tensor:
    """g.sum(0) of a device [rows, cols] tensor in fp32 through esa_column_sum (fixed order); shapes the kernel
    does not take (cols not a multiple of 4, other dtypes) use torch's sum."""
    rows, cols = g.shape
    if g.dtype not in _CODES or cols % 4 or cols < 4:
        return g.float().sum(0)
    g = on_boundary(g.contiguous())
    lib = _lib.load()
    n = ctypes.c_size_t(0)
    _lib.check(lib.esa_column_sum_workspace_size(rows, cols, ctypes.byref(n)), "esa_column_sum_workspace_size")
    ws = torch.empty(int(n.value), dtype=torch.uint8, device=g.device)
    out = torch.empty(cols, dtype=torch.float32, device=g.device)
    _lib.check(lib.esa_column_sum(g.data_ptr(), _CODES[g.dtype], rows, cols, out.data_ptr(), ws.data_ptr(),
                                  ws.numel(), _lib.stream_of(g)), "esa_column_sum")
    return out


_MAX_LINEAR_OUT = 3
_MAX_GRADS = 8
_VP = [ctypes.c_void_p * n for n in range(_MAX_GRADS + 1)]   # host arrays of the C ABI
_CI = [ctypes.c_int * n for n in range(_MAX_GRADS + 1)]
_MAX_FEATURES = 16384


def _wgrad_ok(pairs) -> bool:
    """Whether esa_weight_grad takes every (g, x): fp32 or bf16 device tensors of one dtype, [rows, features]
    contiguous with the same 1 to 2^31 - 1 rows, feature counts multiples of 8 (bf16) or 4 (fp32), 16-byte aligned."""
    g0 = pairs[0][0]
    code = _CODES.get(g0.dtype)
    if code is None or not g0.is_cuda or not 1 <= g0.shape[0] < 2 ** 31:
        return False
    unit = 8 if code == _lib.ESA_BF16 else 4
    for g, x in pairs:
        for t in (g, x):
            if (t.dtype != g0.dtype or t.device != g0.device or t.dim() != 2 or t.shape[0] != g0.shape[0]
                    or t.shape[1] < unit or t.shape[1] % unit or t.shape[1] > _MAX_FEATURES
                    or not t.is_contiguous() or not _aligned(t)):
                return False
    return True


def esa_weight_grad(pairs, bias) -> list[tuple[torch.Tensor, torch.Tensor | None]]:
    """[(g^T x, g.sum(0) or None)] in fp32 for 1-8 (g, x) over the same rows (the shapes ``_wgrad_ok`` accepts)
    through esa_weight_grad; ``bias`` says per pair whether the column sums are wanted."""
    n, (rows, dev) = len(pairs), (pairs[0][0].shape[0], pairs[0][0].device)
    code = _CODES[pairs[0][0].dtype]
    vp, ci = _VP[n], _CI[n]
    o, i = ci(*[g.shape[1] for g, _ in pairs]), ci(*[x.shape[1] for _, x in pairs])
    lib = _lib.load()
    nbytes = ctypes.c_size_t(0)
    _lib.check(lib.esa_weight_grad_workspace_size(rows, n, o, i, code, ctypes.byref(nbytes)),
               "esa_weight_grad_workspace_size")
    ws = torch.empty(max(int(nbytes.value), 16), dtype=torch.uint8, device=dev)
    dw = [torch.empty(g.shape[1], x.shape[1], dtype=torch.float32, device=dev) for g, x in pairs]
    db = [torch.empty(g.shape[1], dtype=torch.float32, device=dev) if b else None for (g, _), b in zip(pairs, bias)]
    _lib.check(lib.esa_weight_grad(rows, n, vp(*[g.data_ptr() for g, _ in pairs]), vp(*[x.data_ptr() for _, x in pairs]),
                                   o, i, code, vp(*[w.data_ptr() for w in dw]), vp(*[_lib.ptr(b) for b in db]),
                                   ws.data_ptr(), ws.numel(), _lib.stream_of(pairs[0][0])), "esa_weight_grad")
    return list(zip(dw, db))


def weight_bias_grads(pairs, need_w, need_b) -> list[tuple[torch.Tensor | None, torch.Tensor | None]]:
    """[(g^T x, g.sum(0))] in fp32 for any (g, x) over the same rows, None where ``need_w`` / ``need_b`` says a
    gradient is not wanted: calls of esa_weight_grad for up to eight where it takes them, else ``weight_grad`` and
    ``column_sum`` one by one (also where the gradients are to be differentiated again: ``weight_grad`` is made
    of torch operations)."""
    wanted = [(p, b) for p, w, b in zip(pairs, need_w, need_b) if w]
    again = torch.is_grad_enabled() and any(t.requires_grad for p, _ in wanted for t in p)
    if wanted and not again:
        if _wgrad_ok([p for p, _ in wanted]):
            got = []
            for i in range(0, len(wanted), _MAX_GRADS):
                part = wanted[i:i + _MAX_GRADS]
                got += esa_weight_grad([p for p, _ in part], [b for _, b in part])
            got = iter(got)
            return [next(got) if w else (None, column_sum(g) if b else None)
                    for (g, _), w, b in zip(pairs, need_w, need_b)]
        if len(pairs) > 1:
            return [weight_bias_grads([p], [w], [b])[0] for p, w, b in zip(pairs, need_w, need_b)]
    return [(weight_grad(g, x) if w else None, column_sum(g) if b else None)
            for (g, x), w, b in zip(pairs, need_w, need_b)]


def _f32_linear_ok(x: torch.Tensor, pairs) -> bool:
    """Whether esa_linear_f32 takes F.linear(x, w, b) for every (w, b): fp32 device tensors, x [rows, K] and
    W [N, K] contiguous, K % 16 == 0, N % 64 == 0, 16-byte aligned rows."""
    if not (x.is_cuda and x.dtype == torch.float32 and x.dim() == 2 and x.is_contiguous() and _aligned(x)):
        return False
    k = x.shape[1]
    if k < 16 or k % 16 or x.shape[0] >= 2 ** 31:
        return False
    for w, b in pairs:
        if not (w.dtype == torch.float32 and w.dim() == 2 and w.shape[1] == k and w.shape[0] % 64 == 0
                and w.is_contiguous() and _aligned(w) and w.device == x.device):
            return False
        if b is not None and not (b.dtype == torch.float32 and b.shape == (w.shape[0],) and b.is_contiguous()
                                  and b.device == x.device):
            return False
    return True


def esa_linear(x: torch.Tensor, pairs) -> list[torch.Tensor]:
    """[F.linear(x, w, b) for (w, b) in pairs] through one launch of esa_linear_f32 (1-3 weights over one fp32
    input of the shapes ``_f32_linear_ok`` accepts; raises otherwise)."""
    pairs = list(pairs)
    if not 1 <= len(pairs) <= _MAX_LINEAR_OUT or not _f32_linear_ok(x, pairs):
        raise ValueError("esa_linear takes 1-3 fp32 weights [N % 64 == 0, K] over a contiguous fp32 x [rows, K], "
                         "K % 16 == 0")
    n = len(pairs)
    ys = [torch.empty(x.shape[0], w.shape[0], dtype=torch.float32, device=x.device) for w, _ in pairs]
    vp = ctypes.c_void_p
    w_arr = (vp * n)(*[w.data_ptr() for w, _ in pairs])
    b_arr = (vp * n)(*[None if b is None else b.data_ptr() for _, b in pairs])
    y_arr = (vp * n)(*[y.data_ptr() for y in ys])
    n_arr = (ctypes.c_int * n)(*[w.shape[0] for w, _ in pairs])
    _lib.check(_lib.load().esa_linear_f32(x.data_ptr(), x.shape[0], x.shape[1], n, w_arr, b_arr, y_arr, n_arr,
                                          _lib.stream_of(x)), "esa_linear_f32")
    return ys


PLAIN, MISH, MAB, ADD = range(4)   # esa_linear_fwd's epilogues


def _gemm_k(k: int) -> bool:
    return 32 <= k <= _MAX_FEATURES and k % 32 == 0


def _gemm_cols(c: int, dtype) -> bool:
    return 8 <= c <= _MAX_FEATURES and c % (8 if dtype == torch.bfloat16 else 4) == 0


def fused_fwd(x, pairs, epilogue=PLAIN, other=None, residual=None, keep=True):
    """esa_linear_fwd: the outputs y_i for PLAIN, else (z or None, result); see the C ABI for the epilogues.
    x [rows, in] and (W, b) of one dtype, contiguous and 16-byte aligned, sizes as ``fused_ok`` accepts."""
    n, rows, dt = len(pairs), x.shape[0], x.dtype
    keep = keep and epilogue != ADD
    ys = [torch.empty(rows, w.shape[0], dtype=dt, device=x.device) if keep else None for w, _ in pairs]
    result = None
    if epilogue != PLAIN:
        result = torch.empty(rows, pairs[0][0].shape[0], dtype=dt if residual is None else torch.float32, device=x.device)
    vp = _VP[n]
    _lib.check(_lib.load().esa_linear_fwd(
        x.data_ptr(), rows, x.shape[1], _CODES[dt], n, vp(*[w.data_ptr() for w, _ in pairs]),
        vp(*[_lib.ptr(b) for _, b in pairs]), vp(*[_lib.ptr(y) for y in ys]),
        _CI[n](*[w.shape[0] for w, _ in pairs]), epilogue, _lib.ptr(other), _lib.ptr(residual),
        _lib.ptr(result), _lib.stream_of(x)), "esa_linear_fwd")
    return ys if epilogue == PLAIN else (ys[0], result)


def fused_dx(pairs, base=None, mish_z=None):
    """esa_linear_dx: [base +] sum of g W over the (g, W) pairs, or (g W) mish'(mish_z)."""
    (g, w), n = pairs[0], len(pairs)
    dx = torch.empty(g.shape[0], w.shape[1], dtype=g.dtype, device=g.device)
    vp = _VP[n]
    _lib.check(_lib.load().esa_linear_dx(
        vp(*[t.data_ptr() for t, _ in pairs]), vp(*[t.data_ptr() for _, t in pairs]), n, g.shape[0],
        _CI[n](*[t.shape[1] for t, _ in pairs]), w.shape[1], _CODES[g.dtype], _lib.ptr(base),
        _lib.ptr(mish_z), dx.data_ptr(), _lib.stream_of(g)), "esa_linear_dx")
    return dx


def fused_ok(x, weights, along: bool) -> bool:
    """Whether esa_linear_fwd (``along``: the contraction runs along the weights' rows) or esa_linear_dx takes
    these sizes and layouts."""
    if not (x.is_cuda and x.dtype in _CODES and x.dim() == 2 and x.shape[0] < 2 ** 31):
        return False
    return all(w.dtype == x.dtype and w.device == x.device and w.is_contiguous() and _aligned(w)
               and _gemm_k(w.shape[1 if along else 0]) and _gemm_cols(w.shape[0 if along else 1], w.dtype)
               for w in weights)


def _library_rate(x, w, fused_passes: bool) -> bool:
    """bf16 products of this size run at a higher rate in the library GEMM, and its call's host time is hidden:
    from 4e10 operations, where the epilogue saves no pass or the contraction is long (129,850 rows: 512 -> 512
    82 vs 101 us, 512 -> 2048 with Mish 513 vs 546, 2048 -> 512 with the residual 363 vs 382; but 512 -> 512 with
    the MAB's residual 235 vs 228, with the block's residual 240 vs 189)."""
    return (x.dtype == torch.bfloat16 and 2 * x.shape[0] * w.numel() >= 4e10
            and (not fused_passes or x.shape[1] >= 1024))


# The Linears of the packed blocks.  ``fused``: the caller's word that esa_linear_fwd / esa_linear_dx take the sizes
# and the weights (``fused_ok`` of both directions).  Rows that come from the caller of the block (the pooling's seeds)
# may start anywhere, so the alignment of the rows is looked at here.

def linear_outputs(x, pairs, fused: bool) -> list[torch.Tensor]:
    """[x W^T + b for (W, b) in pairs]: one launch of esa_linear_fwd, or ``linear_fwd``."""
    if fused and _aligned(x) and not _library_rate(x, pairs[0][0], False):
        return fused_fwd(x, pairs)
    return linear_fwd(x, pairs)


def linear_then_mish(x, w, b, keep: bool, fused: bool):
    """(z = x W^T + b or None, mish(z))."""
    from .activations import mish_forward   # deferred: activations.py takes this module's functions
    if fused and not _library_rate(x, w, False):
        return fused_fwd(x, [(w, b)], MISH, keep=keep)
    (z,) = linear_fwd(x, [(w, b)])
    return z, mish_forward(z)


def linear_then_mab(o, w, b, residual, keep: bool, fused: bool):
    """(z = o W^T + b or None, o + mish(z), in fp32 on top of ``residual`` where that is given)."""
    from .activations import mab_residual_forward, mish_forward
    if fused and not _library_rate(o, w, True):
        return fused_fwd(o, [(w, b)], MAB, o, residual, keep)
    (z,) = linear_fwd(o, [(w, b)])
    return z, mish_forward(z, o) if residual is None else mab_residual_forward(z, o, residual)


def linear_then_add(x, w, b, residual, fused: bool):
    """x W^T + b, rounded, plus the fp32 ``residual``."""
    if fused and not _library_rate(x, w, True):
        return fused_fwd(x, [(w, b)], ADD, residual=residual)[1]
    return linear_fwd(x, [(w, b)])[0] + residual


def input_grad(pairs, fused: bool, base=None, mish_z=None) -> torch.Tensor:
    """[base +] sum of g W over the (g, W) pairs, or (g W) mish'(mish_z); all of one dtype."""
    from .activations import mish_backward
    (g, w) = pairs[0]
    if fused and _aligned(g) and (base is None or _aligned(base)) and not _library_rate(
            g, w, len(pairs) > 1 or base is not None or mish_z is not None):
        return fused_dx(pairs, base, mish_z)
    dx = g.mm(w) if base is None else torch.addmm(base, g, w)
    for g, w in pairs[1:]:
        dx.addmm_(g, w)
    return dx if mish_z is None else mish_backward(mish_z, dx)


def linear_fwd(x: torch.Tensor, pairs) -> list[torch.Tensor]:
    """[F.linear(x, w, b) for (w, b) in pairs] over 2-D x.  Two or three fp32 weights sharing the input (the
    MAB's Q / K / V projections) of the shapes esa_linear_f32 takes run as one launch of it; a single weight,
    and everything else, is F.linear (at one weight the library GEMM is as fast or faster)."""
    pairs = list(pairs)
    if 2 <= len(pairs) <= _MAX_LINEAR_OUT and _f32_linear_ok(x, pairs):
        return esa_linear(x, pairs)
    return [F.linear(x, w, b) for w, b in pairs]


def compute_dtype(x: torch.Tensor, *params: torch.Tensor | None):
    """The dtype a Linear over x computes in: the autocast dtype under autocast (x and the parameters are
    cast to it, as autocast casts F.linear's inputs), else x's dtype when every parameter has it; None for
    mixed dtypes outside autocast (the callers then leave the call to torch's own checks and errors)."""
    if x.is_cuda and torch.is_autocast_enabled("cuda"):
        return torch.get_autocast_dtype("cuda")
    return x.dtype if all(p is None or p.dtype == x.dtype for p in params) else None


_CAST_CACHE: contextvars.ContextVar = contextvars.ContextVar("esa_param_cast_cache", default=None)
_CAST_ALIGN = 128   # elements per cache slot boundary: every cached view starts 256-byte aligned in bf16


def cast_param(p: torch.Tensor | None, dt: torch.dtype):
    """p in dtype dt: the view cached by an enclosing ``param_casts`` when there is one, else p.to(dt)."""
    if p is None or p.dtype == dt:
        return p
    cache = _CAST_CACHE.get()
    if cache is not None:
        hit = cache.get(id(p))
        if hit is not None and hit[0] is p and hit[1].dtype == dt:
            return hit[1]
    return p.to(dt)


@contextlib.contextmanager
def param_casts(params, dt: torch.dtype):
    """Within the block, the Linear functions take the given fp32 device parameters cast to ``dt`` from one
    concatenated cast (a forward under autocast casts every Linear's weight and bias, about a hundred launches of
    a few microseconds for configuration 4's stack; here two or three).  The cached values equal p.to(dt) bit
    for bit; each parameter's slot starts 256-byte aligned."""
    ps, seen = [], set()
    for p in params:
        if p is not None and p.is_cuda and p.dtype == torch.float32 and p.dtype != dt and id(p) not in seen:
            seen.add(id(p))
            ps.append(p)
    if not ps:
        yield
        return
    slots = [p.numel() + -p.numel() % _CAST_ALIGN for p in ps]
    pieces, pad = [], None
    for p, slot in zip(ps, slots):
        pieces.append(p.detach().reshape(-1))
        if slot > p.numel():
            pad = torch.zeros(_CAST_ALIGN, dtype=torch.float32, device=p.device) if pad is None else pad
            pieces.append(pad[:slot - p.numel()])
    cache = {}
    for p, flat in zip(ps, torch.cat(pieces).to(dt).split(slots)):
        flat = flat if flat.numel() == p.numel() else flat[:p.numel()]
        cache[id(p)] = (p, flat if p.dim() == 1 else flat.view(p.shape))
    token = _CAST_CACHE.set(cache)
    try:
        yield
    finally:
        _CAST_CACHE.reset(token)


class _Linear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias):
        w, b = cast_param(weight, x.dtype), cast_param(bias, x.dtype)
        ctx.save_for_backward(x, w)
        ctx.dtypes = (weight.dtype, None if bias is None else bias.dtype)
        return linear_fwd(x, [(w, b)])[0]

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        wdt, bdt = ctx.dtypes
        g = g.contiguous()
        dx = g.mm(w) if ctx.needs_input_grad[0] else None
        ((dw, db),) = weight_bias_grads([(g, x)], [ctx.needs_input_grad[1]],
                                        [bdt is not None and ctx.needs_input_grad[2]])
        return dx, None if dw is None else dw.to(wdt), None if db is None else db.to(bdt)


def linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None = None) -> torch.Tensor:
    """F.linear(x, weight, bias) with the split-K weight gradient (device tensors; CPU tensors use F.linear)."""
    dt = compute_dtype(x, weight, bias) if x.is_cuda else None
    if dt is None:
        return F.linear(x, weight, bias)   # CPU, or mixed dtypes: torch's own type checks and errors
    x = x.to(dt)
    lead = x.shape[:-1]
    y = call(_Linear, x.reshape(-1, x.shape[-1]).contiguous(), weight, bias)
    return y.view(*lead, weight.shape[0])


class _QKV(torch.autograd.Function):
    """q = fc_q(xq), k = fc_k(xk), v = fc_v(xk) (the MAB's V = fc_v(K), esa/mha.py:54-56).  The backward
    accumulates the input gradients of the projections that share an input in the GEMMs themselves
    (addmm with beta = 1) instead of separate add kernels, so self-attention's dx = gq Wq + gk Wk + gv Wv is
    three GEMMs and no add."""

    @staticmethod
    def forward(ctx, xq, xk, wq, bq, wk, bk, wv, bv):
        same = xk is None
        xk_ = xq if same else xk
        dt = xq.dtype
        # the parameters' own dtypes: the backward returns its fp32 gradients in them
        ctx.params = tuple(None if p is None else p.dtype for p in (wq, bq, wk, bk, wv, bv))
        wq, bq, wk, bk, wv, bv = (cast_param(p, dt) for p in (wq, bq, wk, bk, wv, bv))
        if same:
            q, k, v = linear_fwd(xq, [(wq, bq), (wk, bk), (wv, bv)])
        else:
            (q,) = linear_fwd(xq, [(wq, bq)])
            k, v = linear_fwd(xk_, [(wk, bk), (wv, bv)])
        ctx.save_for_backward(xq, None if same else xk, wq, wk, wv)
        ctx.same = same
        return q, k, v

    @staticmethod
    def backward(ctx, gq, gk, gv):
        xq, xk, wq, wk, wv = ctx.saved_tensors
        xk = xq if ctx.same else xk
        gq, gk, gv = gq.contiguous(), gk.contiguous(), gv.contiguous()
        dxq = dxk = None
        if ctx.same:
            if ctx.needs_input_grad[0]:
                dxq = gq.mm(wq)
                dxq.addmm_(gk, wk)
                dxq.addmm_(gv, wv)
        else:
            if ctx.needs_input_grad[0]:
                dxq = gq.mm(wq)
            if ctx.needs_input_grad[1]:
                dxk = gk.mm(wk)
                dxk.addmm_(gv, wv)
        pairs = [(gq, xq), (gk, xk), (gv, xk)]
        need_w = [ctx.needs_input_grad[2 + 2 * i] for i in range(3)]
        need_b = [ctx.params[2 * i + 1] is not None and ctx.needs_input_grad[3 + 2 * i] for i in range(3)]
        if ctx.same:
            parts = weight_bias_grads(pairs, need_w, need_b)
        else:   # the seeds' rows are not the keys'
            parts = (weight_bias_grads(pairs[:1], need_w[:1], need_b[:1])
                     + weight_bias_grads(pairs[1:], need_w[1:], need_b[1:]))
        grads = [dxq, dxk]
        for i, (dw, db) in enumerate(parts):
            grads += [None if dw is None else dw.to(ctx.params[2 * i]),
                      None if db is None else db.to(ctx.params[2 * i + 1])]
        return tuple(grads)


def qkv_projection(fc_q: nn.Linear, fc_k: nn.Linear, fc_v: nn.Linear, xq: torch.Tensor, xk: torch.Tensor):
    """(fc_q(xq), fc_k(xk), fc_v(xk)) on 2-D token rows, with the fused-accumulation backward of _QKV on
    device tensors (``xk is xq`` for self-attention)."""
    params = (fc_q.weight, fc_q.bias, fc_k.weight, fc_k.bias, fc_v.weight, fc_v.bias)
    same = xk is xq
    dt = compute_dtype(xq, xk, *params) if xq.is_cuda else None
    if dt is None:
        return fc_q(xq), fc_k(xk), fc_v(xk)
    xq = xq.to(dt)
    xk_ = None if same else xk.to(dt).contiguous()
    return call(_QKV, xq.contiguous(), xk_, *params)


def hookless(layer: nn.Module) -> bool:
    """True when calling ``layer`` would run no forward hooks or pre-hooks, so its forward may be replaced
    by an equivalent fused call."""
    return not (layer._forward_hooks or layer._forward_pre_hooks)


def apply(layer: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """layer(x), with hook-free nn.Linear layers through ``linear``."""
    if type(layer) is nn.Linear and hookless(layer):
        return linear(x, layer.weight, layer.bias)
    return layer(x)
