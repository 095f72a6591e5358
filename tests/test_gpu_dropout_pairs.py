"""The dense bf16 dropout kernels where a hash is shared by the two keys 2i, 2i + 1: segments that begin at odd
tokens (the kernels walk them from the token before), lengths of a whole group of 128 keys (whose last key then
needs a group of its own), of one key, and around a tile of 32 and a stage of 64.

The oracle's mask is per (query, key) and knows nothing of pairs; the values are at the bf16 bars.  The row staged
before an odd segment belongs to another graph, so that row is then made non-finite: no output of the segment may
change.
"""
import math

import numpy as np
import pytest
import torch

from mind_amd.esa import attention as A
from oracle import attention as OA
from tests._util import assert_bf16_close, cu_from_lengths, grad_scale, seeded_normal

pytestmark = pytest.mark.gpu

ODD = (1, 128, 127, 1, 129, 32, 64, 0, 256, 31)


def _run(device, cu_q, cu_k, q, k, v, g, scale, seed):
    dq, dk = (torch.as_tensor(c.astype(np.int32)).to(device) for c in (cu_q, cu_k))
    dk = dq if cu_q is cu_k else dk
    mq, mk = int(np.diff(cu_q).max()), int(np.diff(cu_k).max())
    t = [x.to(device) for x in (q, k, v, g)]
    kw = {"dropout_p": 0.3, "dropout_seed": seed}
    out, lse = A.attn_fwd(t[0], t[1], t[2], dq, dk, mq, mk, scale, **kw)
    grads = A.attn_bwd(t[3], t[0], t[1], t[2], out, lse, dq, dk, mq, mk, scale, **kw)
    torch.cuda.synchronize()
    return [x.float().cpu() for x in (out, *grads)]


@pytest.mark.parametrize("hd", [16, 24, 32, 64])
@pytest.mark.parametrize("keys", ["self", (3, 65, 128, 0, 31, 96, 1, 0, 127, 33)])
def test_segments_that_begin_at_odd_tokens(device, hd, keys):
    print(f"[dropout-pairs] hd={hd} keys={keys}", flush=True)
    cu_q = np.asarray(cu_from_lengths(ODD))
    cu_k = cu_q if keys == "self" else np.asarray(cu_from_lengths(keys))
    tq, tk, scale, heads = int(cu_q[-1]), int(cu_k[-1]), 1.0 / math.sqrt(hd), 2
    q, g = (seeded_normal((tq, heads, hd), 31 + i, torch.bfloat16) for i in range(2))
    k, v = (seeded_normal((tk, heads, hd), 41 + i, torch.bfloat16) for i in range(2))
    got = _run(device, cu_q, cu_k, q, k, v, g, scale, 77)
    ro, _ = OA.varlen_attention(q, k, v, cu_q, cu_k, scale, dropout=(0.3, 77))
    want = (ro, *OA.varlen_attention_bwd(g, q, k, v, cu_q, cu_k, scale, dropout=(0.3, 77)))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        assert_bf16_close(a, b, grad_scale(b), name)


@pytest.mark.parametrize("hd", [16, 24, 64])
def test_row_before_an_odd_segment_is_not_read(device, hd):
    cu = np.asarray(cu_from_lengths((1, 150)))
    q, k, v, g = (seeded_normal((151, 2, hd), 51 + i, torch.bfloat16) for i in range(4))
    clean = _run(device, cu, cu, q, k, v, g, 0.25, 5)
    for x, bad in ((q, math.inf), (k, math.nan), (v, math.inf), (g, math.nan)):
        x[0] = bad
    dirty = _run(device, cu, cu, q, k, v, g, 0.25, 5)
    for name, a, b in zip(("out", "dq", "dk", "dv"), dirty, clean):
        assert torch.equal(a[1:], b[1:]), name
