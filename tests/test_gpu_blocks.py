"""The packed blocks recorded as one autograd node (mind_amd.esa.blocks) against the separate functions: outputs
and gradients of every input.

Bar, norm-wise per tensor (``_scale``): the two differ in the order of the Linears' sums and in where partial gradients are added
and rounded.  fp32: roundings of 2^-24 per addition, far below 1e-5.  bf16 autocast: a value rounded to bf16 the
other way, or a gradient rounded once more or once less, 2^-9 of its magnitude per rounding, at most four of them on
any path: 2^-7."""
import numpy as np
import pytest
import torch

from mind_amd import generators
from mind_amd.esa import attention, blocks, linear, masked_layers
from mind_amd.esa.packing import EdgeAdjacency, NodeAdjacency

pytestmark = pytest.mark.gpu


def _tokens(device, node, seed=0, graphs=5):
    gb, _ = generators.small_molecules(seed=seed, num_graphs=graphs)
    ei, bm = torch.as_tensor(gb.edge_index).to(device), torch.as_tensor(gb.batch).to(device)
    cls, n = (NodeAdjacency, gb.node_counts.max()) if node else (EdgeAdjacency, gb.edge_counts.max())
    return cls.from_edge_index(ei, bm, gb.num_graphs, int(n) + 3)


def _sab(device, idx, mlp_layers, dropout=0.0, d=64):
    torch.manual_seed(3)
    blk = masked_layers.SABComplete(d, d, 4, dropout, idx, "LN", use_mlp=mlp_layers > 0, mlp_hidden_size=96,
                                    num_mlp_layers=max(mlp_layers, 2), xformers_or_torch_attn="hip").to(device)
    return blk.train()


def _scale(grads, names, i):
    """What gradient i is compared with: itself; a Linear's bias, which sums the rows that its weight (the tensor
    before it) sums against inputs of about 1, with the larger of both (fc_k's is zero but for rounding)."""
    own = float(grads[i].double().norm())
    return max(own, float(grads[i - 1].double().norm())) if names[i].endswith("bias") and ".ln." not in names[i] else own


def _agree(got, want, bar, names):
    for i, (a, b, name) in enumerate(zip(got, want, names)):
        assert a is not None and a.dtype == b.dtype and a.shape == b.shape, name
        assert float((a.double() - b.double()).norm()) <= bar * _scale(want, names, i), name


def _both(one, separate, x, params, g, amp, blk):
    named = {id(p): n for n, p in blk.named_parameters()}
    res = []
    for fn in (one, separate):
        with torch.autocast("cuda", torch.bfloat16, enabled=amp):
            out = fn()
        assert out is not None
        res.append((out, torch.autograd.grad(out, [x] + params, g.to(out.dtype))))
    (o1, g1), (o2, g2) = res
    bar = 2.0 ** -7 if amp else 1e-5
    assert o1.dtype == o2.dtype and float((o1.double() - o2.double()).norm()) <= bar * float(o2.double().norm())
    _agree(g1, g2, bar, ["x"] + [named[id(p)] for p in params])


@pytest.mark.parametrize("amp", [False, True])
@pytest.mark.parametrize("idx,node,mlp_layers,dropout", [(0, False, 2, 0.0), (1, False, 2, 0.0), (1, True, 3, 0.1),
                                                         (0, False, 0, 0.0), (0, False, 2, 0.2)])
def test_sab_block(device, amp, idx, node, mlp_layers, dropout):
    tokens, blk = _tokens(device, node), _sab(device, idx, mlp_layers, dropout)
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    g = torch.randn(tokens.num_tokens, 64, device=device)
    params = [p for n, p in blk.named_parameters() if mlp_layers or "norm_mlp" not in n]
    seeds = []

    def one():
        return blocks.sab_block(blk, x, tokens, idx == 1, dropout, lambda a, seed: seeds.append(seed))

    def separate():
        return masked_layers._sab_separate(blk, x, tokens, seed)

    state = torch.get_rng_state()
    seed = attention.draw_dropout_seed() if dropout else None   # what the block draws from the same state
    torch.set_rng_state(state)
    _both(one, separate, x, params, g, amp, blk)


@pytest.mark.parametrize("amp", [False, True])
@pytest.mark.parametrize("k_seeds,dropout", [(1, 0.0), (4, 0.1)])
def test_pma_block(device, amp, k_seeds, dropout):
    tokens = _tokens(device, False)
    torch.manual_seed(4)
    blk = masked_layers.PMAComplete(64, 4, k_seeds, "LN", dropout=dropout, use_mlp=True, mlp_hidden_size=96,
                                    num_mlp_layers=2, xformers_or_torch_attn="hip").to(device).train()
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    g = torch.randn(tokens.batch_size, k_seeds, 64, device=device)
    state = torch.get_rng_state()
    seed = attention.draw_dropout_seed() if dropout else None
    torch.set_rng_state(state)
    _both(lambda: blocks.pma_block(blk, x, tokens, dropout, None),
          lambda: masked_layers._pma_separate(blk, x, tokens, seed), x, list(blk.parameters()), g, amp, blk)


def test_frozen_parameters_and_input(device):
    tokens, blk = _tokens(device, False), _sab(device, 1, 2)
    for p in list(blk.sab.mab.fc_k.parameters()) + [blk.norm.ln.bias, blk.mlp.mlp[0].weight]:
        p.requires_grad_(False)
    x = torch.randn(tokens.num_tokens, 64, device=device)
    out = blocks.sab_block(blk, x, tokens, True, 0.0, None)
    params = [p for p in blk.parameters() if p.requires_grad]
    got = torch.autograd.grad(out.sum(), params)
    ref = torch.autograd.grad(masked_layers._sab_separate(blk, x, tokens).sum(), params)
    assert all(torch.allclose(a, b, rtol=1e-4, atol=1e-4 * float(b.abs().max())) for a, b in zip(got, ref))
    with torch.no_grad():
        assert torch.equal(blocks.sab_block(blk, x, tokens, True, 0.0, None), out)


def test_differentiated_again_and_not_taken(device):
    tokens, blk = _tokens(device, False), _sab(device, 0, 2)
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    grads = []
    for fn in (lambda: masked_layers._sab_forward_packed(blk, x, tokens), lambda: masked_layers._sab_separate(blk, x, tokens)):
        w = blk.mlp.mlp[2].weight
        (gw,) = torch.autograd.grad(fn().square().sum(), w, create_graph=True)
        assert gw.requires_grad
        grads.append(torch.autograd.grad(gw.square().sum(), w)[0])
    assert torch.allclose(grads[0], grads[1], rtol=1e-4, atol=1e-4 * float(grads[1].abs().max()))
    assert blocks.sab_block(blk, x.bfloat16(), tokens, False, 0.0, None) is None
    with torch.autocast("cuda", torch.float16):
        assert blocks.sab_block(blk, x, tokens, False, 0.0, None) is None
    seen = []
    handle = blk.mlp.register_forward_hook(lambda *a: seen.append(1))
    masked_layers._sab_forward_packed(blk, x, tokens)
    handle.remove()
    assert seen


@pytest.mark.parametrize("amp", [False, True])
def test_strided_and_misaligned_parameters(device, amp):
    """Parameters that the fused products do not take: a transposed weight, a bias off a 16-byte boundary."""
    tokens = _tokens(device, False)
    for which in ("weight", "bias"):
        blk = _sab(device, 0, 2)
        fc = blk.mlp.mlp[0]
        if which == "weight":
            fc.weight = torch.nn.Parameter(fc.weight.detach().t().contiguous().t())
        else:
            fc.bias = torch.nn.Parameter(torch.randn(fc.bias.numel() + 1, device=device)[1:])
        x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
        g = torch.randn(tokens.num_tokens, 64, device=device)
        _both(lambda: blocks.sab_block(blk, x, tokens, False, 0.0, None),
              lambda: masked_layers._sab_separate(blk, x, tokens), x, [blk.mlp.mlp[2].weight, blk.norm.ln.weight], g,
              amp, blk)


def _off_boundary(t):
    """t's values in memory that starts 4 bytes past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, device=t.device)
    return flat[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("amp", [False, True])
def test_rows_off_a_boundary(device, amp):
    """Seeds and output gradients that are views into a larger buffer, as flat parameter and gradient buffers hold
    them: the products over them go where no alignment is asked for."""
    tokens = _tokens(device, False)
    torch.manual_seed(5)
    blk = masked_layers.PMAComplete(64, 4, 2, "LN", use_mlp=False, xformers_or_torch_attn="hip").to(device).train()
    blk.pma.S = torch.nn.Parameter(_off_boundary(blk.pma.S.detach()))
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    g = _off_boundary(torch.randn(tokens.batch_size, 2, 64, device=device))
    params = [p for n, p in blk.named_parameters() if "norm_mlp" not in n]
    _both(lambda: blocks.pma_block(blk, x, tokens, 0.0, None), lambda: masked_layers._pma_separate(blk, x, tokens), x,
          params, g, amp, blk)


@pytest.mark.parametrize("amp", [False, True])
def test_parameters_that_do_not_fit(device, amp):
    """Parameters left on the host or of other shapes raise torch's errors; no kernel takes their addresses."""
    tokens = _tokens(device, False)
    x = torch.randn(tokens.num_tokens, 64, device=device)
    for change in (lambda fc: fc.cpu(), lambda fc: setattr(fc, "weight", torch.nn.Parameter(fc.weight.detach()[:, :32])),
                   lambda fc: setattr(fc, "bias", torch.nn.Parameter(fc.bias.detach()[:32]))):
        for pick in (lambda b: b.sab.mab.fc_o, lambda b: b.mlp.mlp[2]):
            blk = _sab(device, 0, 2)
            change(pick(blk))
            with torch.autocast("cuda", torch.bfloat16, enabled=amp):
                assert blocks.sab_block(blk, x, tokens, False, 0.0, None) is None
                with pytest.raises(RuntimeError):
                    masked_layers._sab_forward_packed(blk, x, tokens)


def _packed(blk, tokens):
    """(the block in one node, through the separate functions): the packed forwards of a SAB or PMA block."""
    one, apart = ((masked_layers._sab_forward_packed, masked_layers._sab_separate) if hasattr(blk, "sab") else
                  (masked_layers._pma_forward_packed, masked_layers._pma_separate))
    return (lambda x: one(blk, x, tokens)), (lambda x: apart(blk, x, tokens))


def _pma(device, mlp=True, dropout=0.0, k_seeds=2):
    torch.manual_seed(5)
    return masked_layers.PMAComplete(64, 4, k_seeds, "LN", dropout=dropout, use_mlp=mlp, mlp_hidden_size=96,
                                     num_mlp_layers=2, xformers_or_torch_attn="hip").to(device).train()


def _used(blk):
    return {n: p for n, p in blk.named_parameters() if blk.use_mlp or "norm_mlp" not in n}


class _Held(torch.nn.Module):
    """A block as a submodule whose forward is its packed one, to be called with other parameters."""

    def __init__(self, blk, fn):
        super().__init__()
        self.blk, self.fn = blk, fn

    def forward(self, x):
        return self.fn(x)


@pytest.mark.parametrize("amp", [False, True])
@pytest.mark.parametrize("pma", [False, True])
def test_differentiated_again_with_other_parameters(device, amp, pma):
    """Parameters substituted for a call (fast weights): a backward that is differentiated again gives the gradients
    of those, and of the weights they are made from."""
    tokens = _tokens(device, False)
    blk = _pma(device) if pma else _sab(device, 1, 3)
    base = {n: (p.detach() * 0.5 + 0.01).requires_grad_(True) for n, p in _used(blk).items()}
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    name, grads, again = "mlp.mlp.2.weight" if pma else "mlp.mlp.4.weight", [], []
    for fn in _packed(blk, tokens):
        fast = {n: p * 1.5 for n, p in base.items()}
        with torch.autocast("cuda", torch.bfloat16, enabled=amp):
            out = torch.func.functional_call(_Held(blk, fn), {"blk." + n: p for n, p in fast.items()}, (x,))
        grads.append(torch.autograd.grad(out.float().sin().sum(), [x, *fast.values(), *base.values()], create_graph=True))
        if not amp:   # the bf16 weight gradients' products (with fp32 results) have no derivative in torch
            gw = grads[-1][1 + list(fast).index(name)]
            again.append(torch.autograd.grad(gw.square().sum(), [fast[name], base[name]]))
    _agree(*grads, 2.0 ** -7 if amp else 1e-5, ["x", *fast, *base])
    if not amp:
        _agree(*again, 2e-5, [name, name])


@pytest.mark.parametrize("pma", [False, True])
def test_differentiated_again_in_another_mode(device, pma):
    """The module leaves training mode between its forward and a backward that is differentiated again: the
    gradients are those of the forward, attention dropout included."""
    tokens = _tokens(device, False)
    blk = _pma(device, dropout=0.3) if pma else _sab(device, 1, 2, 0.3)
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    inputs, grads = [x, *_used(blk).values()], []
    for again in (True, False):
        torch.manual_seed(9)
        out = _packed(blk.train(), tokens)[0](x)
        blk.eval()
        grads.append(torch.autograd.grad(out.sin().sum(), inputs, create_graph=again))
    _agree(*grads, 1e-5, ["x", *_used(blk)])


@pytest.mark.parametrize("amp", [False, True])
@pytest.mark.parametrize("pma", [False, True])
def test_parameters_changed_before_the_backward(device, amp, pma):
    """In-place updates between the forward and its backward of parameters whose values the gradients do not take
    (biases; under autocast the weights, too, of which the cast is kept) leave the gradients as they were.  Where the
    block would have to run again, the change is an error."""
    tokens = _tokens(device, False)
    blk = _pma(device) if pma else _sab(device, 1, 2)
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    used, grads = _used(blk), []
    changed = [p for n, p in used.items() if n.endswith("bias") or (amp and ".ln." not in n)]
    for change in (False, True):
        with torch.autocast("cuda", torch.bfloat16, enabled=amp):
            out = _packed(blk, tokens)[0](x)
        if change:
            with torch.no_grad():
                for p in changed:
                    p.add_(0.5)
            with pytest.raises(RuntimeError, match="modified by an inplace operation"):
                torch.autograd.grad(out.sum(), x, create_graph=True)
        grads.append(torch.autograd.grad(out.sin().sum(), [x, *used.values()]))
    assert all(torch.equal(a, b) for a, b in zip(*grads))


class _Halved(torch.nn.Module):
    """A parametrization that counts how often it is evaluated."""

    def __init__(self):
        super().__init__()
        self.calls = 0

    def forward(self, w):
        self.calls += 1
        return 0.5 * w


@pytest.mark.parametrize("where", ["fc_q", "fc_o", "ln", "S"])
def test_parametrized_parameters(device, where):
    """A parametrized tensor is computed as often as the separate functions compute it (a spectral norm's estimate
    moves with every evaluation) and gets its gradient, also where that is differentiated again."""
    tokens = _tokens(device, False)
    grads, calls = [], []
    for i in range(2):
        blk = _pma(device) if where == "S" else _sab(device, 0, 2)
        owner = {"ln": lambda: blk.norm.ln, "S": lambda: blk.pma}.get(where, lambda: getattr(blk.sab.mab, where))()
        count = _Halved()
        torch.nn.utils.parametrize.register_parametrization(owner, "S" if where == "S" else "weight", count)
        gen = torch.Generator(device).manual_seed(2)
        x = torch.randn(tokens.num_tokens, 64, device=device, generator=gen, requires_grad=True)
        count.calls = 0
        out = _packed(blk, tokens)[i](x)
        calls.append(count.calls)
        params = [p for n, p in blk.named_parameters()]
        grads.append(torch.autograd.grad(out.sin().sum(), [x] + params, create_graph=True))
    assert calls[0] == calls[1]
    _agree(*grads, 1e-5, ["x"] + [n for n, _ in blk.named_parameters()])


def test_replaced_forward_runs(device):
    """A forward set on the MLP itself (as wrappers set it) is called."""
    tokens, blk = _tokens(device, False), _sab(device, 0, 2)
    seen, plain = [], blk.mlp.forward
    blk.mlp.forward = lambda y: seen.append(1) or plain(y)
    _packed(blk, tokens)[0](torch.randn(tokens.num_tokens, 64, device=device))
    assert seen


@pytest.mark.parametrize("amp", [False, True])
@pytest.mark.parametrize("pma", [False, True])
@pytest.mark.parametrize("mlp", [False, True])
def test_output_gradient_off_a_boundary(device, amp, pma, mlp):
    """An output gradient whose memory starts off a 16-byte boundary gives the same gradients as its copy on one."""
    tokens = _tokens(device, False)
    blk = _pma(device, mlp) if pma else _sab(device, 1, 2 * mlp)
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    with torch.autocast("cuda", torch.bfloat16, enabled=amp):
        out = _packed(blk, tokens)[0](x)
    flat = torch.randn(out.numel() + 1, device=device).to(out.dtype)
    g = flat[1:].view(out.shape)
    assert g.data_ptr() % 16
    used = _used(blk)
    got = torch.autograd.grad(out, [x, *used.values()], g, retain_graph=True)
    want = torch.autograd.grad(out, [x, *used.values()], g.clone())
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("amp", [False, True])
@pytest.mark.parametrize("pma", [False, True])
@pytest.mark.parametrize("which", ["one by one", "library"])
def test_large_block_routes(device, monkeypatch, amp, pma, which):
    """What only large blocks take, at a small size: weight gradients computed one by one, products that stay with
    the library."""
    if which == "library":
        monkeypatch.setattr(linear, "_library_rate", lambda *a: True)
    else:
        monkeypatch.setattr(blocks, "_TOGETHER", 0)
    tokens = _tokens(device, False)
    blk = _pma(device) if pma else _sab(device, 1, 3)
    x = torch.randn(tokens.num_tokens, 64, device=device, requires_grad=True)
    g = torch.randn(tokens.batch_size, 2, 64, device=device) if pma else torch.randn(tokens.num_tokens, 64, device=device)
    one, separate = _packed(blk, tokens)
    _both(lambda: one(x), lambda: separate(x), x, list(_used(blk).values()), g, amp, blk)
