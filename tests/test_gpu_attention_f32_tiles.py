"""The tiled fp32 attention kernels at the edges of their tiles: segments of lengths around the 16-token blocks, the
32-token waves, the 64-token stages and the 128-token groups, queries and keys of different lengths, every head dim,
with the edge mask and with dropout, against the fp64 oracle at the fp32 bar of test_gpu_attention_f32 (outputs,
log-sum-exp and gradients within 1e-5 of the largest value)."""
import numpy as np
import pytest
import torch

from mind_amd.esa import attention as A
from oracle import attention as OA
from tests._util import cu_from_lengths
from tests.test_gpu_attention_f32 import _check, _close, _inputs

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 193]


@pytest.mark.parametrize("hd", [16, 24, 32, 64])
def test_self_attention_lengths(device, hd):
    _check(device, EDGES, EDGES, seed=hd, heads=3, hd=hd)


@pytest.mark.parametrize("hd", [16, 64])
def test_cross_attention_lengths(device, hd):
    _check(device, EDGES + [0, 5], EDGES[::-1] + [7, 0], seed=hd + 1, heads=2, hd=hd)


def test_edge_mask_lengths(device):
    rng = np.random.default_rng(0)
    t = sum(EDGES)
    ends = np.repeat(np.arange(len(EDGES)) * 1000, EDGES)   # a node range per segment
    src, dst = (ends + rng.integers(0, 40, t) for _ in range(2))
    _check(device, EDGES, EDGES, seed=5, src=src, dst=dst)


@pytest.mark.parametrize("hd", [16, 24, 64])
def test_dropout_lengths(device, hd):
    p, seed, h, scale = 0.3, 1234567, 2, hd ** -0.5
    cu = cu_from_lengths(EDGES)
    q, k, v, g = _inputs(int(cu[-1]), int(cu[-1]), 3, h, hd)
    qd, kd, vd = (x.to(device).requires_grad_(True) for x in (q, k, v))
    cud, n = torch.as_tensor(cu).to(device), max(EDGES)
    out = A.varlen_attention(qd, kd, vd, cud, cud, n, n, dropout_p=p, dropout_seed=seed, softmax_scale=scale)
    grads = torch.autograd.grad(out, (qd, kd, vd), g.to(device))
    ref, _ = OA.varlen_attention(q, k, v, cu, cu, scale, dropout=(p, seed))
    _close(out.detach().cpu(), ref, "out")
    for got, want, name in zip(grads, OA.varlen_attention_bwd(g, q, k, v, cu, cu, scale, dropout=(p, seed)), "qkv"):
        _close(got.cpu(), want, "d" + name)


@pytest.mark.parametrize("hd,p", [(16, 0.0), (24, 0.2), (64, 0.0)])
@pytest.mark.parametrize("what", ["k", "q", "g"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_edge_mask_nonfinite_row_stays_with_its_neighbours(device, hd, p, what, value):
    """An infinity or a NaN in one token's key, query or output gradient reaches no gradient of a token whose mask
    leaves that token out: those equal the gradients with a finite row there (1e-5 of the largest value: they are
    then added by another instruction)."""
    rng = np.random.default_rng(1)
    length, heads, odd = 200, 2, 77
    src, dst = (rng.integers(0, 40, length) for _ in range(2))
    shares = (src == src[odd]) | (src == dst[odd]) | (dst == src[odd]) | (dst == dst[odd])
    cu = torch.as_tensor(cu_from_lengths([length])).to(device)
    sd, dd = (torch.as_tensor(x.astype(np.int32)).to(device) for x in (src, dst))
    grads = []
    for fill in (0.5, value):
        q, k, v, g = _inputs(length, length, 7, heads, hd)
        {"q": q, "k": k, "g": g}[what][odd, :, 3] = fill
        qd, kd, vd = (x.to(device).requires_grad_(True) for x in (q, k, v))
        out = A.varlen_attention(qd, kd, vd, cu, cu, length, length, edge_src=sd, edge_dst=dd, dropout_p=p,
                                 dropout_seed=11)
        grads.append([x.cpu() for x in torch.autograd.grad(out, (qd, kd, vd), g.to(device))])
    # a token's gradients take in what its neighbours' rows and statistics are: where the odd row spoils those (its
    # neighbours' for a key), the tokens two steps away see it, too
    near = shares
    if what == "k":
        near = np.array([bool((((src == src[i]) | (src == dst[i]) | (dst == src[i]) | (dst == dst[i])) & shares).any())
                         for i in range(length)])
    far, far_q = torch.as_tensor(~near), torch.as_tensor(~shares)
    assert int(far_q.sum()) > 100 and int(far.sum()) > 30
    for name, want, got in zip(("dq", "dk", "dv"), *grads):
        keep = far_q if name == "dq" else far   # dq: the token's own statistics and its keys
        _close(got[keep], want[keep].double(), name)


@pytest.mark.parametrize("hd,p", [(16, 0.0), (24, 0.3), (32, 0.0), (64, 0.0)])
@pytest.mark.parametrize("length", [17, 63, 64, 130])
def test_key_that_no_query_sees(device, hd, p, length):
    """A key whose scores are all -inf (an infinite component against positive ones) has zero probability for every
    query: its own gradients are zeros, the other keys' are those without it, and nothing is a NaN.  (dQ takes the
    key's row times zero, which an infinity makes a NaN.)"""
    odd = length // 2
    rest = [i for i in range(length) if i != odd]
    q, k, v, g = _inputs(length, length, 11, 2, hd)
    q[..., 3] = q[..., 3].abs() + 0.1
    k[odd, :, 3] = -float("inf")
    qd, kd, vd = (x.to(device).requires_grad_(True) for x in (q, k, v))
    cu = torch.as_tensor(cu_from_lengths([length])).to(device)
    out = A.varlen_attention(qd, kd, vd, cu, cu, length, length, dropout_p=p, dropout_seed=3)
    _, dk, dv = torch.autograd.grad(out, (qd, kd, vd), g.to(device))
    assert not out.isnan().any() and not dk.isnan().any() and not dv.isnan().any()
    assert not dk[odd].any() and not dv[odd].any()
    if p == 0.0:
        cur = cu_from_lengths([length]), cu_from_lengths([length - 1])
        want = OA.varlen_attention_bwd(g, q, k[rest], v[rest], *cur, hd ** -0.5)
        for got, ref, name in zip((dk, dv), want[1:], ("dk", "dv")):
            _close(got[rest].cpu(), ref, name)


@pytest.mark.parametrize("hd", [16, 24, 32, 64])
@pytest.mark.parametrize("length", [340, 3000])
def test_output_error_of_long_segments(device, hd, length):
    """The outputs' error stays that of short sums: the products with the values are added over 32 keys and then over
    those sums.  n additions of random signs in a row leave about 2^-24 sqrt(n / 6) of the result, here n = 32 +
    length / 32 (one row of 3,000: 1.3e-6); four units more for the scores (hd products), the exponentials and the
    probabilities' sum."""
    q, k, v, _ = _inputs(length, length, hd, 4, hd)
    cu = cu_from_lengths([length])
    cud = torch.as_tensor(cu).to(device)
    out = A.varlen_attention(*(x.to(device) for x in (q, k, v)), cud, cud, length, length).cpu().double()
    ref, _ = OA.varlen_attention(q, k, v, cu, cu, hd ** -0.5)
    bar = 2.0 ** -24 * (((32 + length / 32) / 6) ** 0.5 + 4)
    assert float((out - ref).norm() / ref.norm()) <= bar
