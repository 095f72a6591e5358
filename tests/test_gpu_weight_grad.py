"""GPU parity of the Linears' weight and bias gradients (esa_weight_grad through mind_amd.esa.linear) against
fp64 products: sizes around the 128 x 128 (and 128 x 256) tiles, the 16- and 32-row stages and the row ranges, one
to three pairs, and the calls that stay with torch's operations.

Bar, elementwise: a value is a sum of fp32 products (bf16 products are exact in fp32) added over a range of rows and
then over the ranges, at most rows additions in all, each within 2^-24 of the magnitudes added so far:
|got - ref| <= (rows + 8) 2^-24 sum_t |g_t x_t|, and the same for the column sums with x = 1."""
import pytest
import torch

from mind_amd.esa import linear as L

pytestmark = pytest.mark.gpu


def _pairs(device, rows, shapes, dtype, seed=0):
    gen = torch.Generator().manual_seed(seed + rows)
    return [(torch.randn(rows, o, generator=gen).to(dtype).to(device),
             torch.randn(rows, i, generator=gen).to(dtype).to(device)) for o, i in shapes]


def _check(pairs, got, bias):
    for (g, x), (dw, db), b in zip(pairs, got, bias):
        g, x = g.double(), x.double()
        unit = (g.shape[0] + 8) * 2.0 ** -24
        assert dw.dtype == torch.float32 and dw.shape == (g.shape[1], x.shape[1])
        assert bool(((dw.double() - g.t() @ x).abs() <= unit * (g.abs().t() @ x.abs())).all())
        assert (db is not None) == b
        if b:
            assert bool(((db.double() - g.sum(0)).abs() <= unit * g.abs().sum(0)).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 32, 33, 127, 128, 255, 257, 4099])
def test_rows(device, dtype, rows):
    pairs = _pairs(device, rows, [(128, 128)], dtype)
    _check(pairs, L.esa_weight_grad(pairs, [True]), [True])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(8, 8), (64, 64), (72, 200), (128, 136), (136, 128), (192, 192), (256, 1024),
                                   (1024, 96)])
def test_features(device, dtype, shape):
    pairs = _pairs(device, 1001, [shape], dtype)
    _check(pairs, L.esa_weight_grad(pairs, [False]), [False])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_three_pairs_share_rows(device, dtype):
    pairs = _pairs(device, 3001, [(64, 128), (200, 128), (128, 40)], dtype)
    got = L.esa_weight_grad(pairs, [True, False, True])
    _check(pairs, got, [True, False, True])
    again = L.esa_weight_grad(pairs, [True, False, True])
    assert all(torch.equal(a[0], b[0]) for a, b in zip(got, again))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [33, 5003])
def test_many_pairs_of_different_shapes(device, dtype, rows):
    """A block's Linears together: eight in a call, two more in a second one, an unwanted weight between them, and
    one the kernel does not take (a bias-only result and a misaligned gradient), which leaves the others to it."""
    shapes = [(64, 128), (200, 136), (128, 40), (8, 8), (256, 64), (64, 256), (136, 128), (128, 128), (40, 72), (72, 8)]
    pairs = _pairs(device, rows, shapes, dtype)
    bias = [i % 3 != 1 for i in range(len(pairs))]
    _check(pairs, L.weight_bias_grads(pairs, [True] * len(pairs), bias), bias)
    (dw, db), *rest = L.weight_bias_grads(pairs[:4], [False] + [True] * 3, [True] * 4)
    assert dw is None and torch.allclose(db, pairs[0][0].float().sum(0), atol=1e-2)
    _check(pairs[1:4], rest, [True] * 3)
    flat = torch.randn(rows * 64 + 1, device=device).to(dtype)
    off = flat[1:].view(rows, 64)
    got = L.weight_bias_grads([(off, pairs[0][1])] + pairs[1:3], [True] * 3, [False] * 3)
    assert torch.allclose(got[0][0].double(), off.double().t() @ pairs[0][1].double(), rtol=2e-2, atol=1.0)
    _check(pairs[1:3], got[1:], [False] * 2)


@pytest.mark.parametrize("shapes", [[(512, 512)] * 3, [(2040, 504)]])
def test_wide_tiles(device, shapes):
    """Enough 128 x 256 tiles and rows for the wide tile, whole and with remainders in rows and features."""
    pairs = _pairs(device, 16411, shapes, torch.bfloat16)
    bias = [i == 0 for i in range(len(shapes))]
    _check(pairs, L.esa_weight_grad(pairs, bias), bias)


def test_other_calls_keep_torch_operations(device):
    """Shapes, dtypes and alignments the kernel does not take, and gradients that are differentiated again."""
    (g, x), = _pairs(device, 300, [(64, 64)], torch.float32)
    for a, b in ((g[:, :63], x), (g[:, :6].contiguous(), x), (g.half(), x.half()), (g[:0], x[:0]),
                 (g.reshape(-1)[1:1 + 64 * 299].view(299, 64), x[:299])):
        assert not L._wgrad_ok([(a, b)])
        ((dw, _),) = L.weight_bias_grads([(a, b)], [True], [False])
        assert torch.allclose(dw.double(), a.double().t() @ b.double(), rtol=0, atol=1e-3 if a.dtype != torch.half else 0.1)
    w = torch.randn(64, 64, device=device, requires_grad=True)
    xr = x.clone().requires_grad_(True)
    (dw,) = torch.autograd.grad((L.linear(xr, w) * g).sum(), w, create_graph=True)
    (dx,) = torch.autograd.grad((dw * w).sum(), xr)   # d/dx sum(w * g^T x) = g w
    assert torch.allclose(dx, g @ w.detach(), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_off_a_boundary(device, dtype):
    """A gradient and an input that start off a 16-byte boundary: weight and bias gradients, the column sum."""
    (g, x), = _pairs(device, 301, [(64, 72)], dtype)
    off = [torch.cat((t.new_zeros(1), t.reshape(-1)))[1:].view(t.shape) for t in (g, x)]
    assert all(t.data_ptr() % 16 for t in off)
    for a, b in (off, (off[0], x), (g, off[1])):
        ((dw, db),) = L.weight_bias_grads([(a, b)], [True], [True])
        _check([(g, x)], [(dw, db)], [True])
    assert torch.equal(L.column_sum(off[0]), L.column_sum(g))


@pytest.mark.parametrize("rows,shape", [(900, (128, 128)), (21752, (256, 128)), (66000, (1024, 1024))])
def test_fp32_error(device, rows, shape):
    """n additions of random signs in a row leave about 2^-24 sqrt(n / 6) of the result.  A bias column is 32 tokens
    (four stages, half of their rows), those sums over a range (up to 4,096 rows, or 512 and those), and at most 512
    ranges in four slices of eights: n = 52 + 64; a weight is the range's rows, or 512 and those sums.  Two units more
    for the last additions."""
    pairs = _pairs(device, rows, [shape], torch.float32)
    ((dw, db),) = L.esa_weight_grad(pairs, [True])
    g, x = (t.double() for t in pairs[0])

    def off(got, ref):
        return float((got.double() - ref).norm() / ref.norm())
    tiles = -(-shape[0] // 128) * -(-shape[1] // 128)
    span = max(128, rows // max(1, 512 // tiles))   # rows of a range
    assert off(db, g.sum(0)) <= 2.0 ** -24 * (((52 + min(span, 4096) / 64) / 6) ** 0.5 + 2)
    assert off(dw, g.t() @ x) <= 2.0 ** -24 * (((span if span <= 4096 else 512 + span / 512) / 6) ** 0.5 + 2)
