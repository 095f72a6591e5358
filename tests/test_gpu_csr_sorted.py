"""The CSR build's sort: keys in order (which it copies), keys one pair away from order at the places the check can
miss, and sizes around its digit widths (8 and 9 bits), tiles (4,096 edges) and the column scan's 1,024 tiles; all
bit-exact against numpy's stable sort."""
import numpy as np
import pytest
import torch

from mind_amd import edges

pytestmark = pytest.mark.gpu


def _check(device, keys, nodes, offset=0):
    buf = torch.as_tensor(np.concatenate([np.zeros(offset, np.int32), keys.astype(np.int32)])).to(device)
    csr = edges.CSR.build(buf[offset:], nodes)
    k = np.where((keys >= 0) & (keys < nodes), keys, nodes)
    assert np.array_equal(csr.perm.cpu().numpy(), np.argsort(k, kind="stable"))
    assert np.array_equal(csr.indptr.cpu().numpy(), np.searchsorted(np.sort(k), np.arange(nodes + 1)))


@pytest.mark.parametrize("nodes", [1, 255, 256, 511, 512, 65535, 70000, 262143, 262144, 1 << 24])
@pytest.mark.parametrize("num", [1, 4095, 4096, 4097, 30001])
def test_digit_widths(device, nodes, num):
    rng = np.random.default_rng(nodes + num)
    keys = rng.integers(-1, nodes + 1, num)
    _check(device, keys, nodes)
    _check(device, np.sort(keys[(keys >= 0) & (keys < nodes)]), nodes, offset=nodes % 2)


@pytest.mark.parametrize("offset", [0, 1])   # 1: not 16-byte aligned, read key by key
@pytest.mark.parametrize("at", [0, 2, 3, 255, 1023, 4095, 4096, 8191, 9998])
def test_one_descent(device, at, offset):
    """Sorted but for keys[at] > keys[at + 1]: inside a lane's four keys, between lanes, waves and tiles."""
    keys = np.arange(10000) // 3 * 2
    keys[at] = keys[at + 1] + 1
    _check(device, keys, 7000, offset)


def test_invalid_keys_among_sorted(device):
    """Invalid keys sort past every valid one: in order only at the end."""
    keys = np.sort(np.random.default_rng(0).integers(0, 1000, 9000))
    for bad in (-1, 1000, 2 ** 31 - 1):
        _check(device, np.concatenate([keys, np.full(500, bad)]), 1000)
        _check(device, np.concatenate([np.full(500, bad), keys]), 1000)


@pytest.mark.parametrize("tiles", [1024, 1025])
@pytest.mark.parametrize("ordered", [False, True])
def test_column_scan_limit(device, tiles, ordered):
    keys = np.random.default_rng(tiles).integers(0, 100000, tiles * 4096 - 5)
    _check(device, np.sort(keys) if ordered else keys, 100000)
