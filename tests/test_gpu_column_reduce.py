"""The one-launch reduction of column partials (bias gradients, LayerNorm parameter gradients) where its 32 slices
and 32-column blocks are ragged: no rows, fewer partials than slices, one more than a multiple of them, column counts
around a block.  Whole-number inputs: every fp32 partial sum is exact (below 2^24), so the results are too."""
import pytest
import torch

from mind_amd.esa.layer_norm import layer_norm
from mind_amd.esa.linear import column_sum

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [4, 28, 32, 36, 1028])
@pytest.mark.parametrize("rows", [0, 1, 31 * 32, 31 * 32 + 1, 33 * 32, 1024 * 32 + 7])
def test_column_sum_is_exact_on_whole_numbers(device, rows, cols):
    print(f"[column-reduce] {rows} x {cols}", flush=True)
    x = torch.randint(-8, 9, (rows, cols), generator=torch.Generator().manual_seed(rows + cols)).float()
    assert torch.equal(column_sum(x.to(device)).cpu(), x.double().sum(0).float())


@pytest.mark.parametrize("features", [4, 36, 512])
@pytest.mark.parametrize("rows", [0, 1, 125, 129, 5003])
def test_layer_norm_parameter_gradients(device, rows, features):
    """Rows alternating +a, -a have mean 0 and xhat = +-1 up to eps, so both sums are whole numbers before it."""
    print(f"[column-reduce] layer norm {rows} x {features}", flush=True)
    g = torch.Generator().manual_seed(rows + features)
    sign = torch.ones(features)
    sign[1::2] = -1
    x = (1024.0 * sign).repeat(rows, 1).to(device).requires_grad_(True)
    ln = torch.nn.LayerNorm(features).to(device)
    dy = torch.randint(-8, 9, (rows, features), generator=g).float()
    layer_norm(x, ln)[0].backward(dy.to(device))
    assert torch.equal(ln.bias.grad.cpu(), dy.double().sum(0).float())
    # rstd = 1 / 1024 within 2 roundings (eps / 1024^2 = 1e-11), then rows fp32 additions
    bar = (2 * 2.0 ** -23 + rows * 2.0 ** -24) * dy.abs().double().sum(0)
    assert bool(((ln.weight.grad.cpu().double() - (dy.double() * sign).sum(0)).abs() <= bar).all())
