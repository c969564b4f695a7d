"""The work that users of this framework have it do, as measurable cases.

Every case is one pass of a user's program through the public entry points of the ``fastgl`` package: a mini-batch
sampled (``FusedMapSampler``, ``DataLoader``, the per-hop operators), a training or inference step of a model over
freshly sampled blocks, or a layer's operators over a block that the user brings along.  Graphs are seeded R-MAT graphs,
features are N(0, 1), weights the layers' own initialisation; everything is made from the seed and lives on the GPU.

Fields of a case: ``kind`` (sample | hops | loader | train | infer | block | graph), the graph (``nodes``, R-MAT
``draws`` before mirroring and deduplication), the mini-batch (``batch`` seeds, ``fanouts`` in the reference's order: the
last one expands the seeds), and for the layers ``model``, ``dim`` -> ``hidden`` -> ``classes`` and ``dtype``.
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "fastgl-ae_amd"))  # the repository's root is the working folder
import fastgl  # noqa: E402

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
HEADS = 4        # attention heads of the GAT cases, as in train.py
IN_EPOCH = 8     # mini-batches of one pass of the "loader" cases


def listed():
    mid = dict(nodes=2_400_000, draws=36_000_000)
    return [
        # -- sampling: all hops of one mini-batch, sizes read back by the host ------------------------------------
        # a small graph and batch: latency and launches count (the benchmark's smallest workload)
        dict(name="sample_small", kind="sample", nodes=100_000, draws=1_500_000, batch=1024, fanouts="15,10,5", deterministic=False),
        # an ordinary graph (the size of the trainer's default), full batch
        dict(name="sample_mid", kind="sample", batch=8192, fanouts="15,10,5", deterministic=False, **mid),
        # the benchmark's headline graph: 111 M nodes, 1.7 G edges
        dict(name="sample_large", kind="sample", nodes=111_000_000, draws=900_000_000, batch=8192, fanouts="15,10,5", deterministic=False),
        # deep sampling for a five-layer model with reproducible gradients (ordered transposed blocks)
        dict(name="sample_deep", kind="sample", batch=1000, fanouts="10,10,10,10,10", deterministic=True, **mid),
        # the reference's own loop: sample_node and transfer_edge_id per hop, its default fanouts and batch
        dict(name="hops_dropin", kind="hops", batch=8000, fanouts="5,10,15", **mid),
        # the prefetching loader over a stretch of an epoch, its short last batch among them
        dict(name="loader_epoch", kind="loader", batch=2000, fanouts="15,10,5", **mid),
        # -- models over freshly sampled blocks -----------------------------------------------------------------
        # online inference for a handful of seeds: the smallest call
        dict(name="infer_gcn_small", kind="infer", model="gcn", nodes=100_000, draws=1_500_000, batch=100, fanouts="10,10", dim=100,
             hidden=64, classes=47, dtype="f32"),
        # GraphSAGE in bf16, the first layer gathering straight from the resident feature table
        dict(name="train_sage_bf16", kind="train", model="sage", batch=8192, fanouts="15,10,5", dim=128, hidden=256, classes=47,
             dtype="bf16", **mid),
        # the trainer's default sizes with GCN
        dict(name="train_gcn", kind="train", model="gcn", batch=8192, fanouts="15,10,5", dim=100, hidden=256, classes=16, dtype="f32", **mid),
        # attention: the reference's default hidden size and a batch of a thousand
        dict(name="train_gat", kind="train", model="gat", batch=1000, fanouts="15,10,5", dim=100, hidden=64, classes=16, dtype="f32", **mid),
        # -- layers over blocks that the user brings (drop-in operators; the transposed block is theirs to build) -----
        # GIN over 8192 rows of 25 neighbours out of 200 K rows of 602 columns (the aggregation benchmark's widest rows)
        dict(name="block_gin_602", kind="block", rows=8192, cols=200_000, per_row=25, dim=602, hidden=256, dtype="f32"),
        # full-graph GCN: the whole graph as one block, from its edge list; hub rows of tens of thousands of entries
        dict(name="graph_gcn", kind="graph", dim=100, hidden=64, dtype="f32", **mid),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["sample", "sample", "hops", "loader", "train", "train", "train", "infer", "block", "graph"])
    if kind == "block":
        c = dict(kind=kind, rows=_log_uniform(rng, 500, 20_000), cols=_log_uniform(rng, 5_000, 200_000), per_row=rng.randint(1, 30),
                 dim=rng.choice([rng.randint(16, 602), 64, 128, 256]), hidden=_log_uniform(rng, 16, 256), dtype=rng.choice(["f32", "bf16"]))
        return c
    nodes = _log_uniform(rng, 20_000, 2_400_000)
    c = dict(kind=kind, nodes=nodes, draws=int(nodes * rng.uniform(5, 15)))
    if kind == "graph":
        c.update(dim=rng.randint(16, 100), hidden=_log_uniform(rng, 16, 64), dtype=rng.choice(["f32", "bf16"]))
        return c
    c.update(batch=_log_uniform(rng, 50, 8192), fanouts=rng.choice(["15,10,5", "5,10,15", "10,10", "25,10", "10,10,10", "10,25"]))
    if kind == "sample":
        c["deterministic"] = rng.random() < 0.3
        if not c["deterministic"] and c["batch"] <= 1000 and rng.random() < 0.3:
            c["fanouts"] = "10,10,10,10,10"
    if kind == "loader":
        c["batch"] = min(c["batch"], 4000)
    if kind in ("train", "infer"):
        c.update(model=rng.choice(["gcn", "gin", "gat", "sage"]), dim=rng.choice([rng.randint(16, 300), 100, 128, 256]),
                 hidden=rng.choice([rng.randint(16, 256), 64, 128, 256]), classes=_log_uniform(rng, 2, 172), dtype=rng.choice(["f32", "bf16"]))
        if c["model"] == "gat":  # (attention coefficients are float32)
            c.update(dtype="f32", hidden=min(c["hidden"], 64))
    return c


def _fanouts(case):
    return [int(f) for f in case["fanouts"].split(",")]


def _sampler(case, seed):
    """The graph, a sampler on it and enough training seeds for one stretch of an epoch."""
    edge_ptr, edge_src = fastgl.graph.rmat_csr(case["nodes"], case["draws"], seed=seed, device=DEV)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    n = case["batch"] if case["kind"] != "loader" else (IN_EPOCH - 1) * case["batch"] + (case["batch"] + 1) // 2
    n = min(n, case["nodes"])
    seeds = torch.randperm(case["nodes"], generator=gen, device=DEV)[:n].int()
    sampler = fastgl.FusedMapSampler(_fanouts(case), rng_seed=seed, fused=case["kind"] != "hops",
                                     deterministic=bool(case.get("deterministic", False)), transposed="none" if case["kind"] == "infer" else "inner")
    return sampler.set_graph(edge_ptr, edge_src), seeds, gen


def _model(case, seed):
    torch.manual_seed(seed)
    args = (case["dim"], case["hidden"], case["classes"], len(_fanouts(case)))
    if case["model"] == "sage":
        m = fastgl.SAGE(*args)
    elif case["model"] == "gat":
        m = fastgl.GAT(*args, None, 0.0, heads=HEADS)
    else:
        m = {"gcn": fastgl.GCN, "gin": fastgl.GIN}[case["model"]](*args, None, True, 0.0)
    return m.to(DEV).to(DTYPES[case["dtype"]])


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "block":
        gen = torch.Generator(device=DEV).manual_seed(seed)
        n, k = case["rows"], case["per_row"]
        dt = DTYPES[case["dtype"]]
        s["edge_ptr"] = torch.arange(n + 1, dtype=torch.int32, device=DEV) * k
        s["src"] = torch.randint(0, case["cols"], (n * k,), generator=gen, dtype=torch.int32, device=DEV)
        s["feat"] = torch.randn((case["cols"], case["dim"]), generator=gen, device=DEV).to(dt)
        s["weight"] = ((torch.rand((case["dim"], case["hidden"]), generator=gen, device=DEV) * 2 - 1) / case["hidden"] ** 0.5).to(dt)
        s["d_out"] = torch.randn((n, case["hidden"]), generator=gen, device=DEV).to(dt)
        return s
    if kind == "graph":
        edge_ptr, edge_src = fastgl.graph.rmat_csr(case["nodes"], case["draws"], seed=seed, device=DEV)
        gen = torch.Generator(device=DEV).manual_seed(seed)
        n, dt = case["nodes"], DTYPES[case["dtype"]]
        deg = edge_ptr[1:] - edge_ptr[:-1]
        s["src"] = edge_src
        s["dst"] = torch.repeat_interleave(torch.arange(n, dtype=torch.int32, device=DEV), deg)
        s["longest"] = int(deg.max())
        s["feat"] = torch.randn((n, case["dim"]), generator=gen, device=DEV).to(dt)
        s["weight"] = ((torch.rand((case["dim"], case["hidden"]), generator=gen, device=DEV) * 2 - 1) / case["hidden"] ** 0.5).to(dt)
        s["d_out"] = torch.randn((n, case["hidden"]), generator=gen, device=DEV).to(dt)
        return s
    s["sampler"], s["seeds"], gen = _sampler(case, seed)
    if kind in ("sample", "hops", "loader"):
        s["packed"] = torch.full((IN_EPOCH if kind == "loader" else 1, _bounds(case)), -1, dtype=torch.int32, device=DEV)
    if kind == "loader":
        s["loader"] = fastgl.DataLoader(None, s["seeds"], s["sampler"], batch_size=case["batch"], shuffle=True, prefetch_factor=2, seed=seed)
    if kind in ("train", "infer"):
        s["feat"] = torch.randn((case["nodes"], case["dim"]), generator=gen, device=DEV).to(DTYPES[case["dtype"]])
        s["label"] = torch.randint(0, case["classes"], (case["nodes"],), generator=gen, device=DEV)
        s["model"] = _model(case, seed)
    return s


def _bounds(case):
    """What the packed arrays of one mini-batch take at most, in words: node bounds n, edge bounds e per hop."""
    n, words = case["batch"], 0
    for f in reversed(_fanouts(case)):
        words += n + 1 + n * f                                  # offsets and local ids
        more = min(n + n * f, case["nodes"] + case["batch"])
        words += more + 1 + (2 * n * f if case.get("deterministic", False) else 0)  # the transposed block
        n = more
    return words + n


def _pack(buf, input_nodes, blocks, transposed, ordered):
    """The mini-batch in one buffer of fixed size, as a program with static shapes (a captured graph, another process)
    takes it; returns the pieces' lengths."""
    pieces = [input_nodes] + [x for b in blocks for x in (b.edge_ptr, b.src_local)]
    if transposed:
        # the transposed inner blocks that come with a mini-batch: their row pointers, and -- where the sampler was asked for
        # an order inside the rows -- their entries
        for b in blocks[1:]:
            pieces += b.transposed(edge_ids=True) if ordered else b.transposed()[:1]
    sizes = [p.numel() for p in pieces]
    torch.cat(pieces, out=buf[:sum(sizes)])
    return sizes


def _logits(s, blocks, input_nodes):
    case = s["case"]
    if case["model"] == "sage":
        return s["model"](blocks, s["feat"], input_nodes=input_nodes)
    return s["model"](blocks, s["feat"].index_select(0, input_nodes), neighbor_list=_fanouts(case))


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "sample":
        input_nodes, _, blocks = s["sampler"].sample_blocks(None, s["seeds"])
        return [_pack(s["packed"][0], input_nodes, blocks, True, case["deterministic"]), s["packed"]]
    if kind == "hops":
        input_nodes, _, blocks = s["sampler"].sample_blocks(None, s["seeds"])
        return [_pack(s["packed"][0], input_nodes, blocks, False, False), s["packed"]]
    if kind == "loader":
        sizes = []
        for i, (input_nodes, _, blocks) in enumerate(s["loader"]):
            sizes += _pack(s["packed"][i], input_nodes, blocks, False, False)[:1]
        return [sizes, s["packed"]]
    if kind == "infer":
        input_nodes, _, blocks = s["sampler"].sample_blocks(None, s["seeds"])
        with torch.no_grad():
            return _logits(s, blocks, input_nodes)
    if kind == "train":
        input_nodes, output_nodes, blocks = s["sampler"].sample_blocks(None, s["seeds"])
        fastgl.transpose_blocks(blocks[1:])
        labels = s["label"].index_select(0, output_nodes)
        logits = _logits(s, blocks, input_nodes)
        loss = torch.nn.functional.cross_entropy(logits.float(), labels)
        s["model"].zero_grad()
        loss.backward()
        return [logits.detach()] + [p.grad for p in s["model"].parameters() if p.grad is not None]
    if kind == "block":  # GIN layer, forward and backward (MA_Function_GIN's calls)
        out, tmp = fastgl.forwaed_gin(s["edge_ptr"], s["src"], s["feat"], s["weight"], case["per_row"], case["rows"])
        return [out] + fastgl.backward_gin(s["edge_ptr"], s["src"], s["d_out"], s["weight"], tmp, case["cols"])
    # the whole graph, from its edge list: a GCN layer's calls, forward and backward
    n = case["nodes"]
    raw = fastgl.cal_deg(s["dst"], n)
    edge_ptr = fastgl.exclusive_sum(raw)
    dst_norm = raw.clamp(min=1)
    src_norm = fastgl.cal_deg(s["src"], n).clamp(min=1)
    out = fastgl.forward_gcn(edge_ptr, s["src"], src_norm, dst_norm, s["feat"], s["weight"], s["longest"], n)
    return out + fastgl.backward_gcn(edge_ptr, s["src"], dst_norm, src_norm, s["d_out"], s["weight"], s["feat"])


def _counts(case):
    """Node counts before each hop and after the last, and edge counts per hop, of the case's first mini-batch."""
    sampler, seeds, _ = _sampler(dict(case, kind="sample"), 0)
    _, _, blocks = sampler.sample_blocks(None, seeds)
    blocks = blocks[::-1]
    return [b.num_dst_nodes() for b in blocks] + [blocks[-1].num_src_nodes()], [b.num_edges() for b in blocks]


def _sampling_bytes(nodes, edges, transposed):
    # per hop: the seeds' row offsets (two of eight bytes), the picked neighbour ids in, the block out (offsets, local ids),
    # the unique ids out; the inner hops' transposed blocks
    total = sum(16 * n + 4 * e + 4 * n + 4 * e for n, e in zip(nodes, edges)) + 4 * nodes[-1]
    if transposed:
        total += sum(4 * n + 8 * e for n, e in zip(nodes[1:-1], edges[:-1]))
    return total


def work(case):
    kind = case["kind"]
    sz = 4 if case.get("dtype", "f32") == "f32" else 2
    if kind in ("block", "graph"):
        if kind == "block":
            n_dst, n_src, e = case["rows"], case["cols"], case["rows"] * case["per_row"]
            seen = int(n_src * (1 - (1 - 1 / n_src) ** e))  # distinct rows among e uniform draws
            first = n_dst
        else:
            edge_ptr, _ = fastgl.graph.rmat_csr(case["nodes"], case["draws"], seed=0, device=DEV)
            n_dst = n_src = seen = case["nodes"]
            e = int(edge_ptr[-1])
            first = n_src
        d, h = case["dim"], case["hidden"]
        # features and edges in, output, gradients of the features and of the weights out
        size = seen * d * sz + (4 * e if kind == "block" else 8 * e) + 2 * n_dst * h * sz + n_src * d * sz + 3 * d * h * sz
        gathered = d if kind == "block" else h
        return {"bytes": size, "flops": 3 * 2 * first * d * h + 2 * 2 * e * gathered}
    nodes, edges = _counts(case)
    size = _sampling_bytes(nodes, edges, kind in ("sample", "train", "loader"))
    if kind == "loader":
        size *= IN_EPOCH - 0.5
    if kind not in ("train", "infer"):
        return {"bytes": size, "flops": 0}
    # layers from the outermost block in: gathered rows in once, rows out once; the products; backward the same again
    n_hops = len(edges)
    heads = HEADS if case["model"] == "gat" else 1
    dims = [case["dim"]] + [case["hidden"] * heads] * (n_hops - 1) + [case["classes"]]
    flops, size = 0, size + nodes[-1] * case["dim"] * sz
    for layer in range(n_hops):
        hop = n_hops - 1 - layer
        n_dst, e, d, h = nodes[hop], edges[hop], dims[layer], dims[layer + 1]
        products = n_dst * (2 if case["model"] == "sage" else 1)
        times = 1 if kind == "infer" else 2 if layer == 0 else 3
        flops += times * 2 * products * d * h + 2 * e * min(d, h) * (1 if kind == "infer" or layer == 0 else 2)
        size += n_dst * h * sz * (1 if kind == "infer" else 3) + d * h * sz * (1 if kind == "infer" else 2)
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """Measured against the same passes in float64 (worst output): f32 steps are off by 3e-6 (gradients of the first layer's
    weights), the widest block's weight gradient by 1.6e-6, the full graph's weight gradient -- sums over all nodes -- by 8e-6;
    bf16 steps by 2e-2 to 8e-2 (rounded hidden values change which units a rectifier passes).  Four times the f32 figures;
    for bf16 less than a comparison with float64 would need, since both sides round at the same places."""
    if case["kind"] in ("sample", "hops", "loader"):
        return "exact"
    if case["dtype"] == "bf16":
        return {"rel": 2e-2 if case["kind"] == "train" else 1e-2}
    return {"rel": 3e-5 if case["kind"] == "graph" else 1.2e-5}
