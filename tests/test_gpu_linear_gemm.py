"""GPU parity of the Linears with their epilogues and of their input gradients (esa_linear_fwd / esa_linear_dx through
mind_amd.esa.linear) against fp64: rows and features around the 64- and 128-wide tiles, contractions of one to
several stages, one to three weights or terms, every epilogue, and the sizes that stay with the library.

Bars, elementwise.  A product is a sum of K fp32 terms (bf16 products are exact in fp32): (K + 4) 2^-24 times the
sum of the terms' magnitudes, plus the result's rounding (u = 2^-8 in bf16, 2^-24 in fp32, relative).  Mish and its
slope are evaluated in fp32 (a few 2^-24 relative, hardware exp and reciprocal: 2^-20 of |z| + 1 taken) from z as it is
stored, and |mish'| < 1.1 carries the product's error."""
import pytest
import torch
from torch.nn import functional as F

from mind_amd import edges
from mind_amd.esa import linear as L

pytestmark = pytest.mark.gpu

U = {torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}
DTYPES = [torch.bfloat16, torch.float32]


def _randn(device, *shape, dtype=torch.float32, seed=0):
    gen = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=gen).to(dtype).to(device)


def _product(x, w, b=None):
    """(value, bound on the unrounded fp32 sum's error)."""
    x, w = x.double(), w.double()
    ref, size = x @ w.t(), x.abs() @ w.abs().t()
    if b is not None:
        ref, size = ref + b.double(), size + b.double().abs()
    return ref, (x.shape[1] + 4) * 2.0 ** -24 * size


def _near(got, ref, bound):
    assert got.shape == ref.shape
    assert bool(((got.double() - ref).abs() <= bound).all()), float(((got.double() - ref).abs() - bound).max())


def _forward(device, rows, k, n, dtype, bias=True):
    x, w = _randn(device, rows, k, dtype=dtype), _randn(device, n, k, dtype=dtype, seed=1)
    b = _randn(device, n, dtype=dtype, seed=2) if bias else None
    o, r = _randn(device, rows, n, dtype=dtype, seed=3), _randn(device, rows, n, seed=4)
    assert L.fused_ok(x, [w], True)
    u, (ref, err) = U[dtype], _product(x, w, b)
    (y,) = L.fused_fwd(x, [(w, b)])
    _near(y, ref, err + u * ref.abs())
    fine = 2.0 ** -20 * (y.double().abs() + 1)   # mish from the stored z
    m = F.mish(y.double())
    for keep in (True, False):
        z, h = L.fused_fwd(x, [(w, b)], L.MISH, keep=keep)
        assert torch.equal(z, y) if keep else z is None
        _near(h, m, fine + u * m.abs())
    _, s = L.fused_fwd(x, [(w, b)], L.MAB, o)
    full = o.double() + m
    _near(s, full, fine + 2 * u * full.abs())
    _, s = L.fused_fwd(x, [(w, b)], L.MAB, o, r)
    assert s.dtype == torch.float32
    _near(s, r.double() + full, fine + 2 * u * full.abs() + 2.0 ** -23 * (r.double().abs() + full.abs()))
    _, s = L.fused_fwd(x, [(w, b)], L.ADD, residual=r)
    _near(s, r.double() + y.double(), 2.0 ** -23 * (r.double().abs() + y.double().abs()))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [1, 31, 32, 33, 63, 64, 65, 129, 1000])
def test_forward_rows(device, dtype, rows):
    _forward(device, rows, 64, 72, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k,n", [(32, 8), (64, 64), (96, 136), (128, 200), (192, 128), (1024, 256)])
def test_forward_features(device, dtype, k, n):
    _forward(device, 197, k, n, dtype, bias=k != 64)


@pytest.mark.parametrize("rows,k,n", [(12345, 64, 1024), (9000, 1024, 4096)])
def test_forward_wide_tiles(device, rows, k, n):
    """bf16 at sizes that take the 128 x 128 and 128 x 256 tiles, with rows left over."""
    _forward(device, rows, k, n, torch.bfloat16)


@pytest.mark.parametrize("dtype", DTYPES)
def test_three_outputs(device, dtype):
    x = _randn(device, 333, 96, dtype=dtype)
    pairs = [(_randn(device, n, 96, dtype=dtype, seed=n), _randn(device, n, dtype=dtype) if n != 64 else None)
             for n in (64, 200, 128)]
    for y, (w, b) in zip(L.fused_fwd(x, pairs), pairs):
        ref, err = _product(x, w, b)
        _near(y, ref, err + U[dtype] * ref.abs())


def _gradient(device, rows, terms, k, dtype):
    pairs = [(_randn(device, rows, n, dtype=dtype, seed=n), _randn(device, n, k, dtype=dtype, seed=n + 1)) for n in terms]
    base, z = _randn(device, rows, k, dtype=dtype, seed=5), _randn(device, rows, k, dtype=dtype, seed=6)
    assert L.fused_ok(pairs[0][0], [w for _, w in pairs], False)
    parts = [_product(g, w.t()) for g, w in pairs]
    ref, err, u = sum(p[0] for p in parts), len(terms) * sum(p[1] for p in parts), U[dtype]
    _near(L.fused_dx(pairs), ref, err + u * ref.abs())
    full = ref + base.double()
    _near(L.fused_dx(pairs, base=base), full, err + (u + 2.0 ** -23) * (full.abs() + base.double().abs()))
    zd = z.double().requires_grad_(True)
    (slope,) = torch.autograd.grad(F.mish(zd).sum(), zd)
    got = ref * slope
    _near(L.fused_dx(pairs, mish_z=z), got, 1.1 * (err + u * ref.abs()) + 2.0 ** -19 * ref.abs() + u * got.abs())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,terms,k", [(1, [32], 8), (64, [64], 64), (65, [96], 72), (129, [128, 128, 128], 128),
                                          (300, [32, 160], 200), (1000, [256], 136)])
def test_gradients(device, dtype, rows, terms, k):
    _gradient(device, rows, terms, k, dtype)


@pytest.mark.parametrize("rows,terms,k", [(12345, [64], 1024), (17000, [512, 512], 2048)])
def test_gradients_wide_tiles(device, rows, terms, k):
    _gradient(device, rows, terms, k, torch.bfloat16)


def test_other_sizes_use_the_library(device):
    x, w = _randn(device, 50, 40), _randn(device, 24, 40)   # a contraction that is no whole stage
    assert not L.fused_ok(x, [w], True)
    z, h = L.linear_then_mish(x, w, None, True, False)
    assert torch.equal(z, F.linear(x, w)) and torch.allclose(h, F.mish(z), atol=1e-6)
    assert torch.allclose(L.input_grad([(_randn(device, 50, 24), w)], False), _randn(device, 50, 24) @ w, atol=1e-5)
    assert not L.fused_ok(x.half(), [w.half()], True) and not L.fused_ok(x, [w.t().contiguous().t()], True)
    empty = torch.empty(0, 64, device=device)
    (y,) = L.linear_outputs(empty, [(_randn(device, 64, 64), None)], True)
    assert y.shape == (0, 64)


@pytest.mark.parametrize("out_features", [40, 64])   # 40: the library's product, 64: esa_linear_dx
def test_edge_linear_input_gradient_is_rounded_once(device, out_features):
    """dx = [gs | gd] [W_s; W_d] over the per-node sums of the edge gradients: one rounding of the sum of both halves.
    The halves nearly cancel here (W_d = -W_s but for a tenth), so a rounding of the first alone would show."""
    n, e, f = 300, 3000, 64
    x = _randn(device, n, f, dtype=torch.bfloat16).requires_grad_(True)
    ws = _randn(device, out_features, f, seed=1)
    w = torch.cat((ws, -ws + 0.1 * _randn(device, out_features, f, seed=2)), 1).bfloat16().requires_grad_(True)
    gen = torch.Generator().manual_seed(7)
    src = torch.randint(n, (e,), generator=gen).int().to(device)
    g = _randn(device, e, out_features, dtype=torch.bfloat16, seed=3)
    out = edges.edge_token_linear(x, src, src, w, None)
    (dx,) = torch.autograd.grad(out, x, g)
    csr = edges.CSR.build(src, n)
    gs = edges.segment_sum_csr(g, csr.indptr, csr.perm)
    wd = w.detach()
    ref, err = _product(torch.cat((gs, gs), 1), torch.cat((wd[:, :f], wd[:, f:]), 0).t())
    _near(dx, ref, err + U[torch.bfloat16] * ref.abs())


@pytest.mark.parametrize("widths", [(512, 512, 512), (32, 160, 64), (2048,)])
def test_fp32_error_of_long_contractions(device, widths):
    """fp32 adds 128 values of a term at a time, and then those sums: n additions of random signs in a row leave about
    2^-24 sqrt(n / 6) of the result, here n = 128 + length / 128 (one row of 1,536: 9.5e-7), and one rounding more."""
    gen = torch.Generator().manual_seed(sum(widths))
    rows, cols = 1000, 96
    pairs = [(torch.randn(rows, k, generator=gen).to(device), torch.randn(k, cols, generator=gen).to(device))
             for k in widths]
    ref = sum(g.double() @ w.double() for g, w in pairs)
    bar = 2.0 ** -24 * (((128 + sum(widths) / 128) / 6) ** 0.5 + 1)
    assert float((L.fused_dx(pairs).double() - ref).norm() / ref.norm()) <= bar
    (g, w), = pairs[:1]
    ref = g.double() @ w.double()
    assert float((L.fused_fwd(g, [(w.t().contiguous(), None)])[0].double() - ref).norm() / ref.norm()) <= bar
