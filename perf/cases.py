"""The work that programs have this framework do, as cases: what a pass runs, through the public entry points.

Four kinds of case:

  attention  one attention layer's ``varlen_attention`` over a packed batch of graphs, forward and backward, dense
             or with the edge-adjacency mask or the node adjacency (whose plan is built for each batch)
  esa        the ESA module on packed edge tokens: the batch's descriptor, the blocks, the pooled graph
             embeddings; the forward alone (``train`` false, no autograd) or with every gradient; ``amp`` is
             bf16 autocast over fp32 parameters
  tokens     edge-token construction: ``linear`` false is the gather of both endpoints' features and the sum of
             edge rows back to the nodes (with its CSR); true is the edge MLP's first Linear, forward and backward
  reduce     the atom encoder's edge -> node reductions: a CSR by source with a 1-D sum and a minimum, a CSR by
             target with a sum of feature rows

The graphs are the synthetic molecules and protein-like chains of ``mind_amd.generators``: which graphs a batch
holds is the case's, their order in the batch and all features and weights come from the seed.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch
from torch.nn import functional as F

from mind_amd import generators
from mind_amd.edges import CSR, edge_gather, edge_token_linear, scatter_add, scatter_min
from mind_amd.esa.attention import edge_plan, node_plan, varlen_attention
from mind_amd.esa.masked_layers import ESA
from mind_amd.esa.packing import EdgeAdjacency

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
DEV = "cuda"


def _attention(mask, graphs, size, heads, head_dim, dtype="bf16", dropout=0.0, pick=0):
    return {"kind": "attention", "mask": mask, "graphs": graphs, "size": size, "pick": pick, "heads": heads,
            "head_dim": head_dim, "dtype": dtype, "dropout": dropout}


def _esa(graphs, size, layers, dim, heads, mlp, seeds, train, amp, pick=0):
    return {"kind": "esa", "graphs": graphs, "size": size, "pick": pick, "layers": layers, "dim": dim, "heads": heads,
            "mlp": mlp, "seeds": seeds, "train": train, "amp": amp}


def listed():
    return [
        # A property server's small request: eight molecules through a trained fp32 model; launches and latency.
        dict(_esa("molecules", 8, "MSP", 128, 8, 256, 1, False, False), name="molecules-infer-fp32"),
        # Fine-tuning that model at full precision on an ordinary batch: fp32 attention in both directions.
        dict(_esa("molecules", 64, "MSP", 128, 8, 256, 1, True, False), name="molecules-train-fp32"),
        # The unmasked layer of the pretraining model (16 heads of 16) on a batch of protein-like graphs.
        dict(_attention("none", "proteins", 32, 16, 16), name="dense-16x16"),
        # The same layer of the wide models (512 / 8 heads).
        dict(_attention("none", "proteins", 24, 8, 64, pick=1), name="dense-8x64"),
        # A layer trained with attention dropout (192 / 8 heads, p = 0.08).
        dict(_attention("none", "proteins", 32, 8, 24, dropout=0.08, pick=2), name="dense-8x24-dropout"),
        # The masked layer in edge mode on a token-budget batch: plan, forward, backward.
        dict(_attention("edge", "budget", 65536, 16, 16), name="edge-mask-16x16"),
        # The masked layer in node mode: the adjacency's plan, forward, backward.
        dict(_attention("node", "nodes", 65536, 16, 16), name="node-mask-16x16"),
        # One masked and one unmasked block with pooling in a bf16 train step (256 / 16 heads).
        dict(_esa("proteins", 24, "MSP", 256, 16, 1024, 4, True, True, pick=3), name="blocks-train-bf16"),
        # The whole encoder in a bf16 train step on the largest token budget (512 / 32 heads, MLP 2048).
        dict(_esa("budget", 131072, "MMSSMMSSP", 512, 32, 2048, 4, True, True), name="stack-train-bf16"),
        # Edge tokens from node features and edge outputs back to the nodes, on a large graph: memory traffic.
        {"kind": "tokens", "linear": False, "nodes": 1 << 18, "edges": 1 << 22, "features": 256, "out": 256,
         "dtype": "fp32", "name": "gather-scatter-fp32"},
        # The edge MLP's first Linear over both endpoints' features, forward and backward.
        {"kind": "tokens", "linear": True, "nodes": 28274, "edges": 129850, "features": 256, "out": 512,
         "dtype": "bf16", "name": "edge-linear-bf16"},
        # The atom encoder's reductions over a large batch's edges (128 radial features).
        {"kind": "reduce", "nodes": 1 << 17, "edges": (1 << 20) + 12345, "features": 128, "dtype": "fp32",
         "name": "encoder-reduce-fp32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "esa", "esa", "tokens", "reduce"])
    pick = rng.randrange(1 << 20)
    if kind == "attention":
        mask = rng.choice(["none", "none", "edge", "node"])
        heads, head_dim = rng.choice([(16, 16), (8, 16), (32, 16), (8, 24), (16, 32), (8, 32), (8, 64)])
        dropout = rng.choice([0.0, 0.0, 0.0, 0.08])
        # fp32 modules are the small-molecule models'; the protein batches run bf16
        if rng.random() < 0.2:
            return _attention(mask if mask != "node" else "none", "molecules", _log(rng, 4, 96), heads, head_dim,
                              "fp32", dropout, pick)
        if mask == "node":
            return _attention(mask, "nodes", _log(rng, 2000, 65536), heads, head_dim, "bf16", dropout, pick)
        if mask == "edge":
            return _attention(mask, "budget", _log(rng, 4000, 80000), heads, head_dim, "bf16", dropout, pick)
        graphs = rng.choice(["proteins", "molecules"])
        return _attention(mask, graphs, _log(rng, 1, 32) if graphs == "proteins" else _log(rng, 8, 256), heads,
                          head_dim, "bf16", dropout, pick)
    if kind == "esa":
        train = rng.random() < 0.6
        if rng.random() < 0.5:
            return _esa("molecules", _log(rng, 1, 96), rng.choice(["MSP", "MMSP", "SP"]), 128, 8, 256,
                        rng.choice([1, 2, 4]), train, rng.random() < 0.3, pick)
        dim, heads = rng.choice([(256, 16), (512, 32), (512, 16), (192, 8)])
        return _esa("proteins", _log(rng, 2, 32), rng.choice(["MSP", "MP", "SP"]), dim, heads, 4 * dim,
                    rng.choice([1, 4]), train, True, pick)
    dtype = rng.choice(["fp32", "bf16"])
    if kind == "tokens":
        linear = rng.random() < 0.4
        edges = _log(rng, 3000, 500000 if linear else 4000000)
        return {"kind": "tokens", "linear": linear, "nodes": max(64, int(edges / rng.uniform(3.0, 17.0))),
                "edges": edges, "features": rng.choice([64, 128, 192, 256]), "out": rng.choice([128, 256, 512]),
                "dtype": dtype}
    edges = _log(rng, 3000, 2000000)
    return {"kind": "reduce", "nodes": max(64, int(edges / rng.uniform(3.0, 17.0))), "edges": edges,
            "features": rng.choice([16, 64, 128]), "dtype": dtype}


# ------------------------------------------------------------------------------------------------ the batches

@functools.lru_cache(maxsize=32)
def _graphs(graphs, size, pick):
    """The case's graphs in their generator's order."""
    if graphs == "molecules":
        return generators.small_molecules(seed=pick, num_graphs=size)[0]
    if graphs == "proteins":
        return generators.protein_like(seed=pick, num_graphs=size)
    return generators.protein_budget(seed=pick, token_budget=size, count="nodes" if graphs == "nodes" else "edges")


@functools.lru_cache(maxsize=32)
def _counts(graphs, size, pick):
    """(tokens, sum of L^2, mask entries in edge mode, edges, nodes) of a batch."""
    gb = _graphs(graphs, size, pick)
    counts = gb.node_counts if graphs == "nodes" else gb.edge_counts
    deg_s = np.bincount(gb.edge_index[0], minlength=gb.pos.shape[0]).astype(np.int64)
    deg_t = np.bincount(gb.edge_index[1], minlength=gb.pos.shape[0]).astype(np.int64)
    deg = deg_s + deg_t   # each edge meets the others at its two endpoints; its reverse is met at both
    n = gb.pos.shape[0]
    key, rev = gb.edge_index[0] * n + gb.edge_index[1], gb.edge_index[1] * n + gb.edge_index[0]
    nnz = int((deg * (deg - 1)).sum() - np.isin(rev, key).sum())
    return int(counts.sum()), int((counts.astype(np.int64) ** 2).sum()), nnz, int(gb.num_tokens), n


def _shuffled(case, seed):
    """(edge_index [2, E], graph of each node, nodes per graph, edges per graph): the case's graphs in an order of
    the seed, as a shuffling loader gives them."""
    gb = _graphs(case["graphs"], case["size"], case["pick"])
    order = np.random.default_rng(seed).permutation(gb.num_graphs)
    nc, ec = gb.node_counts[order], gb.edge_counts[order]
    n0 = np.concatenate([[0], np.cumsum(gb.node_counts)])[:-1][order]
    e0 = np.concatenate([[0], np.cumsum(gb.edge_counts)])[:-1][order]
    new_n0 = np.concatenate([[0], np.cumsum(nc)])[:-1]
    within = np.arange(int(ec.sum())) - np.repeat(np.cumsum(ec) - ec, ec)
    ei = gb.edge_index[:, np.repeat(e0, ec) + within] + np.repeat(new_n0 - n0, ec)
    return ei, np.repeat(np.arange(gb.num_graphs), nc), nc, ec


def _cu(counts):
    return torch.as_tensor(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32))


def _csr(ei, nodes):
    """Rows by source, ascending targets, as int32."""
    order = np.lexsort((ei[1], ei[0]))
    indptr = np.concatenate([[0], np.cumsum(np.bincount(ei[0], minlength=nodes))])
    return torch.as_tensor(indptr.astype(np.int32)), torch.as_tensor(ei[1][order].astype(np.int32))


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)

    def randn(*shape, dtype=torch.float32):
        return torch.randn(*shape, device=DEV, generator=gen).to(dtype)

    if case["kind"] == "attention":
        ei, _, nc, ec = _shuffled(case, seed)
        counts = nc if case["mask"] == "node" else ec
        t, dt = int(counts.sum()), DTYPES[case["dtype"]]
        s = {"case": case, "cu": _cu(counts).to(DEV), "max": int(counts.max()), "dropout_seed": 1000003 * (seed + 1)}
        for name in ("q", "k", "v"):
            s[name] = randn(t, case["heads"], case["head_dim"], dtype=dt).requires_grad_(True)
        s["g"] = randn(t, case["heads"], case["head_dim"], dtype=dt)
        if case["mask"] == "edge":
            s["src"], s["dst"] = (torch.as_tensor(x.astype(np.int32)).to(DEV) for x in ei)
        elif case["mask"] == "node":
            s["indptr"], s["indices"] = (x.to(DEV) for x in _csr(ei, t))
        return s
    if case["kind"] == "esa":
        ei, bm, nc, ec = _shuffled(case, seed)
        d, layers = case["dim"], case["layers"]
        with torch.random.fork_rng(devices=[]):
            torch.manual_seed(seed)
            model = ESA(num_outputs=case["seeds"], dim_output=d, dim_hidden=[d] * len(layers),
                        num_heads=[case["heads"]] * len(layers), layer_types=layers, xformers_or_torch_attn="hip",
                        use_mlps=True, mlp_hidden_size=case["mlp"], num_mlp_layers=2, mlp_type="standard").to(DEV)
        x = randn(int(ec.sum()), d)
        s = {"case": case, "model": model.train(case["train"]), "ei": torch.as_tensor(ei).to(DEV),
             "bm": torch.as_tensor(bm).to(DEV), "graphs": len(ec), "max": int(ec.max()), "x": x}
        if case["train"]:
            x.requires_grad_(True)
            s["g"] = randn(len(ec), d)
            s["params"] = [p for p in model.parameters()]
        return s
    n, e, f, dt = case["nodes"], case["edges"], case["features"], DTYPES[case["dtype"]]
    block = min(512, n)   # a neighbourhood: both ends of an edge lie in one run of nodes; edges in target order
    dst = torch.randint(n, (e,), device=DEV, generator=gen).sort().values
    src = (dst // block * block + torch.randint(block, (e,), device=DEV, generator=gen)).clamp_(max=n - 1)
    s = {"case": case, "src": src.int(), "dst": dst.int()}
    if case["kind"] == "reduce":
        s["dist"], s["rows"] = torch.rand(e, device=DEV, generator=gen).mul_(8).to(dt), randn(e, f, dtype=dt)
    elif case["linear"]:
        s["x"] = randn(n, f, dtype=dt).requires_grad_(True)
        s["w"] = randn(case["out"], 2 * f).mul_(1 / math.sqrt(2 * f)).to(dt).requires_grad_(True)
        s["b"] = randn(case["out"]).mul_(0.1).to(dt).requires_grad_(True)
        s["g"] = randn(e, case["out"], dtype=dt)
    else:
        s["x"], s["y"] = randn(n, f, dtype=dt), randn(e, f, dtype=dt)
    return s


# ------------------------------------------------------------------------------------------------ one pass

def run(s):
    case = s["case"]
    if case["kind"] == "attention":
        mask = {}
        if case["mask"] == "edge":
            mask["edge_plan"] = edge_plan(s["src"], s["dst"], s["cu"])
        elif case["mask"] == "node":
            mask = {"adj_indptr": s["indptr"], "adj_indices": s["indices"],
                    "adj_plan": node_plan(s["indptr"], s["indices"], s["cu"])}
        out = varlen_attention(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["max"], s["max"],
                               dropout_p=case["dropout"], dropout_seed=s["dropout_seed"], **mask)
        dq, dk, dv = torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["g"])
        return {"out": out, "dq": dq, "dk": dk, "dv": dv}
    if case["kind"] == "esa":
        model, x = s["model"], s["x"]
        with torch.set_grad_enabled(case["train"]), torch.autocast("cuda", torch.bfloat16, enabled=case["amp"]):
            tokens = EdgeAdjacency.from_edge_index(s["ei"], s["bm"], s["graphs"], s["max"])
            emb, enc = model.forward_packed(x, tokens)
        if not case["train"]:
            return {"emb": emb, "enc": enc}
        grads = torch.autograd.grad(emb, [x] + s["params"], s["g"].to(emb.dtype))
        return _grouped(emb, grads)
    src, dst, n = s["src"], s["dst"], case["nodes"]
    if case["kind"] == "reduce":
        by_src = CSR.build(src, n)
        total = scatter_add(s["dist"], src, dim_size=n, csr=by_src)
        near, arg = scatter_min(s["dist"], src, dim_size=n, csr=by_src)
        rows = scatter_add(s["rows"], dst, dim_size=n, csr=CSR.build(dst, n))
        return {"total": total, "near": near, "arg": arg, "rows": rows}
    if case["linear"]:
        out = edge_token_linear(s["x"], src, dst, s["w"], s["b"])
        dx, dw, db = torch.autograd.grad(out, (s["x"], s["w"], s["b"]), s["g"])
        return {"out": out, "dx": dx, "dw": dw, "db": db}
    return {"tokens": edge_gather(s["x"], src, dst), "sums": scatter_add(s["y"], dst, dim_size=n)}


def _grouped(emb, grads):
    """The embeddings and every gradient: the matrices one by one, the vectors (biases, norms) as one, as a
    program that reduces or clips gradients buckets its small ones."""
    return {"emb": emb, "dx": grads[0], "matrices": [g for g in grads[1:] if g.dim() > 1],
            "vectors": torch.cat([g for g in grads[1:] if g.dim() == 1])}


# ------------------------------------------------------------------------------------------------ what it takes

def work(case):
    if case["kind"] == "attention":
        t, sq, edge_nnz, edges, nodes = _counts(case["graphs"], case["size"], case["pick"])
        d, size = case["heads"] * case["head_dim"], 4 if case["dtype"] == "fp32" else 2
        pairs = {"none": sq, "edge": edge_nnz, "node": edges}[case["mask"]]
        index = {"none": 0, "edge": 8 * t, "node": 4 * (t + edges)}[case["mask"]]
        return {"bytes": 8 * t * d * size + index, "flops": 14 * d * pairs}
    if case["kind"] == "esa":
        t, sq, nnz, edges, nodes = _counts(case["graphs"], case["size"], case["pick"])
        d, m, graphs = case["dim"], case["mlp"], _graphs(case["graphs"], case["size"], case["pick"]).num_graphs
        times = 3 if case["train"] else 1   # a product's gradients are two more of it
        attn = (14 if case["train"] else 4) * d
        flops = params = 0
        for kind in case["layers"]:
            rows = case["seeds"] * graphs if kind == "P" else t
            gemm = 2 * rows * (2 * d * d + 2 * d * m) + 2 * t * 2 * d * d
            flops += times * gemm + attn * {"M": nnz, "S": sq, "P": case["seeds"] * t}[kind]
            params += 4 * d * d + 2 * d * m
        return {"bytes": 4 * (2 * t * d + (2 if case["train"] else 1) * params), "flops": flops}
    n, e, f, size = case["nodes"], case["edges"], case["features"], 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "reduce":
        return {"bytes": e * (8 + size + f * size) + n * (2 * size + 8 + f * size), "flops": e * (f + 2)}
    if case["linear"]:
        o = case["out"]
        # out written, its gradient read; the node-level products forward and twice backward
        return {"bytes": 2 * e * o * size + 2 * n * f * size + 4 * f * o * size + 8 * e,
                "flops": 3 * 2 * n * 2 * o * f + 4 * e * o}
    return {"bytes": e * 3 * f * size + 2 * n * f * size + 8 * e, "flops": e * f}


def tolerance(case):
    """About four times the error against 64 bits: bf16 operands and outputs round at 2^-9."""
    if case["kind"] == "attention":
        return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 5e-6, "max": 1e-3}
    if case["kind"] == "esa":
        if case["amp"]:   # 1.1e-2 after nine layers, 9e-3 after three
            return {"rel": 3e-2 if len(case["layers"]) > 4 else 2.5e-2, "max": 1.0}
        return {"rel": 1e-5, "max": 2e-3}
    if case["kind"] == "reduce":
        return {"rel": 1e-6, "max": 1e-4} if case["dtype"] == "fp32" else {"rel": 8e-3}
    if case["linear"]:
        return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 5e-6, "max": 1e-3}
    return {"rel": 1e-6, "max": 1e-4} if case["dtype"] == "fp32" else {"rel": 8e-3}


# ------------------------------------------------------------------------------------------------ in 64 bits

def _fmix32(h):
    """MurmurHash3's 32-bit finalizer on int64 values that hold 32 bits."""
    for shift, mul in ((16, 0x85EBCA6B), (13, 0xC2B2AE35)):
        h = ((h ^ (h >> shift)) * mul) & 0xFFFFFFFF
    return h ^ (h >> 16)


def _kept(p, seed, heads, q0, q1, k0, k1):
    """The scaled keep mask [heads, queries, keys] of attention dropout, from its definition: the keys 2i and
    2i + 1 take the low and high 16 bits of fmix32(row(q, head) ^ col(i)), kept at or above thr."""
    thr = min(math.floor(float(np.float32(p)) * 65536 + 0.5), 65535)
    q = torch.arange(q0, q1, device=DEV)[None, :] * heads + torch.arange(heads, device=DEV)[:, None]
    k = torch.arange(k0, k1, device=DEV)
    row = _fmix32((seed & 0xFFFFFFFF) ^ _fmix32(q & 0xFFFFFFFF))
    col = _fmix32(((seed >> 32) ^ 0x9E3779B9) & 0xFFFFFFFF ^ _fmix32(k >> 1))
    bits = _fmix32(row[:, :, None] ^ col[None, None, :])
    return (((bits >> (16 * (k & 1))) & 0xFFFF) >= thr).double() * (65536 / (65536 - thr))


def _attend(q, k, v, allowed, kept, scale):
    """softmax(q k^T scale) v of one graph, heads first [H, L, hd]; a query without a key gives 0."""
    a = (q @ k.transpose(1, 2).contiguous()) * scale
    if allowed is not None:
        a = a.masked_fill(~allowed, -math.inf)
        p = torch.softmax(a, -1)
        p = torch.where(allowed.any(-1)[:, None], p, torch.zeros_like(p))
    else:
        p = torch.softmax(a, -1)
    return (p if kept is None else p * kept) @ v


def _share(src, dst):
    """Which edges of one graph share an endpoint, an edge with itself left out."""
    m = ((src[:, None] == src) | (src[:, None] == dst) | (dst[:, None] == src) | (dst[:, None] == dst))
    return m.fill_diagonal_(False)


def _over_graphs(q, k, v, cu_q, cu_k, allowed_of, kept_of):
    """[T, H, hd] attention graph by graph; nothing of a graph's scores is kept for the backward."""
    outs = []
    for b in range(len(cu_k) - 1):
        q0, q1, k0, k1 = cu_q[b], cu_q[b + 1], cu_k[b], cu_k[b + 1]

        def one(qq, kk, vv, b=b, at=(q0, q1, k0, k1)):
            return _attend(qq.transpose(0, 1), kk.transpose(0, 1), vv.transpose(0, 1), allowed_of(b),
                           kept_of(*at), 1 / math.sqrt(qq.shape[-1])).transpose(0, 1)

        outs.append(torch.utils.checkpoint.checkpoint(one, q[q0:q1], k[k0:k1], v[k0:k1], use_reentrant=False))
    return torch.cat(outs)


def _exact_attention(case, s):
    cu = s["cu"].tolist()
    q, k, v = (s[n].detach().double().requires_grad_(True) for n in ("q", "k", "v"))
    if case["mask"] == "edge":
        def allowed(b):
            return _share(s["src"][cu[b]:cu[b + 1]], s["dst"][cu[b]:cu[b + 1]])
    elif case["mask"] == "node":
        rows = torch.repeat_interleave(torch.arange(cu[-1], device=DEV), s["indptr"].diff())

        def allowed(b):
            e0, e1 = (int(s["indptr"][cu[i]]) for i in (b, b + 1))
            m = torch.zeros(cu[b + 1] - cu[b], cu[b + 1] - cu[b], dtype=torch.bool, device=DEV)
            m[rows[e0:e1] - cu[b], s["indices"][e0:e1].long() - cu[b]] = True
            return m
    else:
        def allowed(b):
            return None

    def kept(*at):
        return _kept(case["dropout"], s["dropout_seed"], case["heads"], *at) if case["dropout"] else None

    out = _over_graphs(q, k, v, cu, cu, allowed, kept)
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), s["g"].double())
    return {"out": out, "dq": dq, "dk": dk, "dv": dv}


def _exact_esa(case, s):
    p = {k: v.detach().double().requires_grad_(case["train"]) for k, v in s["model"].named_parameters()}
    src, dst = s["ei"]
    counts = torch.bincount(s["bm"][src], minlength=s["graphs"]).tolist()
    cu = [0] + np.cumsum(counts).tolist()
    x = s["x"].detach().double().requires_grad_(case["train"])
    heads, d = case["heads"], case["dim"]

    def linear(name, t):
        return F.linear(t, p[name + ".weight"], p[name + ".bias"])

    def norm(name, t):
        return F.layer_norm(t, (d,), p[name + ".ln.weight"], p[name + ".ln.bias"], 1e-8)

    def mlp(name, t):
        return linear(name + ".mlp.mlp.2", F.mish(linear(name + ".mlp.mlp.0", t)))

    def mab(name, qs, ks, cu_q, masked):
        q, k, v = (linear(name + n, t).view(-1, heads, d // heads)
                   for n, t in ((".fc_q", qs), (".fc_k", ks), (".fc_v", ks)))
        o = _over_graphs(q, k, v, cu_q, cu, lambda b: _share(src[cu[b]:cu[b + 1]], dst[cu[b]:cu[b + 1]])
                         if masked else None, lambda *at: None).reshape(-1, d)
        return o + F.mish(linear(name + ".fc_o", o))

    with torch.set_grad_enabled(case["train"]):
        h = x
        for i, kind in enumerate(case["layers"][:-1]):   # the last layer is the pooling
            at = "encoder.%d" % i
            n = norm(at + ".norm", h)
            h = n + mab(at + ".sab.mab", n, n, cu, kind == "M")
            h = h + mlp(at, norm(at + ".norm_mlp", h))
        enc = h + x
        n, seeds, graphs = norm("decoder.0.norm", enc), case["seeds"], s["graphs"]
        q = p["decoder.0.pma.S"].reshape(seeds, d).repeat(graphs, 1)
        h = mab("decoder.0.pma.mab", q, n, [seeds * b for b in range(graphs + 1)], False)
        h = h + mlp("decoder.0", norm("decoder.0.norm_mlp", h))
        emb = F.mish(linear("decoder_linear", h.view(graphs, seeds, d).mean(1)))
    if not case["train"]:
        return {"emb": emb, "enc": enc}
    return _grouped(emb, torch.autograd.grad(emb, [x] + list(p.values()), s["g"].double()))


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "attention":
        return _exact_attention(case, s)
    if case["kind"] == "esa":
        return _exact_esa(case, s)
    src, dst, n = s["src"].long(), s["dst"].long(), case["nodes"]
    if case["kind"] == "reduce":
        dist, rows = s["dist"].double(), s["rows"].double()
        zero = dist.new_zeros(n)
        return {"total": zero.index_add(0, src, dist), "arg": None,
                "near": zero.scatter_reduce(0, src, dist, "amin", include_self=False),
                "rows": rows.new_zeros(n, rows.shape[1]).index_add_(0, dst, rows)}
    if case["linear"]:
        x, w, b = (s[k].detach().double().requires_grad_(True) for k in ("x", "w", "b"))
        out = F.linear(torch.cat((x[src], x[dst]), 1), w, b)
        dx, dw, db = torch.autograd.grad(out, (x, w, b), s["g"].double())
        return {"out": out, "dx": dx, "dw": dw, "db": db}
    x, y = s["x"].double(), s["y"].double()
    return {"tokens": torch.cat((x[src], x[dst]), 1), "sums": y.new_zeros(n, y.shape[1]).index_add_(0, dst, y)}
