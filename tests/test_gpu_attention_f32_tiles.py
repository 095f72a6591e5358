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
