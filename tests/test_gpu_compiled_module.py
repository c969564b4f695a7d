"""The compiled torch extension module `fastgl` (fastgl-ae_amd/csrc/fastgl_module.cpp, built by
`make -C fastgl-ae_amd/csrc module`): the reference's own call sequences -- the sampler's layer loop
(FusedMapSampler.py:72-107) and a GCN / GIN layer's operator calls (GraphConv.py:91-98, 26, 37, 109, 132) --
driven through it, checked against the oracle.  The module is loaded from its file under a private name: in this
test process the name `fastgl` belongs to the Python package."""
import glob
import importlib.util
import os

import numpy as np
import pytest
import torch

from conftest import ROOT

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ext():
    paths = glob.glob(os.path.join(ROOT, "fastgl-ae_amd", "fastgl_ext", "fastgl*.so"))
    if not paths:
        pytest.fail("the compiled module is not built: make -C fastgl-ae_amd/csrc module")
    spec = importlib.util.spec_from_file_location("fastgl", paths[0])
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def rel_err(got, want):
    want = np.asarray(want, dtype=np.float64)
    return np.abs(got.double().cpu().numpy() - want).max() / max(np.abs(want).max(), 1e-30)


def reference_layer_loop(ext, edge_src, edge_dst, edge_ptr, nodes_num, seed_nodes, fanouts):
    """FusedMapSampler.sample_blocks of the reference, statement for statement, with a (src, dst, n_src, n_dst)
    tuple where it builds a DGL block."""
    raw_seed_nodes = seed_nodes.int().clone()
    seed_nodes_acc = seed_nodes.clone()
    blocks = []
    dst_nodes = seed_nodes.size(0)
    for block_index, fanout in enumerate(reversed(fanouts)):
        src_edges_out, dst_edges_out, edge_num = ext.sample_node(edge_src, edge_dst, edge_ptr, seed_nodes_acc.int(), dst_nodes, fanout)
        edge_nums = src_edges_out.size(0)
        assert int(edge_num.item()) == edge_nums
        if block_index == 0:
            dst_edges_unique = raw_seed_nodes
        else:
            dst_edges_unique = seed_nodes_acc
        if block_index == 0:
            output_nodes = raw_seed_nodes
        max_src_num = nodes_num if (fanout * dst_edges_unique.size(0) > nodes_num) else (fanout * dst_edges_unique.size(0))
        src_global = src_edges_out.clone()
        src_edges, dst_edges, seed_nodes_acc = ext.transfer_edge_id(src_edges_out, dst_edges_out, dst_edges_unique,
                                                                    dst_nodes, dst_nodes + edge_nums, max_src_num, edge_nums)
        assert src_edges.data_ptr() == src_edges_out.data_ptr() and dst_edges.data_ptr() == dst_edges_out.data_ptr()  # in place
        blocks.insert(0, (src_edges, dst_edges, seed_nodes_acc.size(0), dst_edges_unique.size(0), src_global))
        dst_nodes = seed_nodes_acc.size(0)
    return seed_nodes_acc, output_nodes, blocks


def test_sampler_loop_and_layers_through_the_compiled_module(cuda, oracle, small_graph, ext):
    print("compiled module: sampler loop + layer operators", flush=True)
    import fastgl
    assert ext.abi_version() == fastgl.lib().fgl_abi_version()
    indptr, indices = small_graph
    n = indptr.size - 1
    # the trainer's CSR: int32 offsets (train_fastgl.py:228-230) -- and int64, which this build also takes
    for ptr_dtype in (np.int32, np.int64):
        edge_ptr = torch.from_numpy(indptr.astype(ptr_dtype)).to(cuda)
        edge_src = torch.from_numpy(indices).to(cuda)
        edge_dst = torch.repeat_interleave(torch.arange(n, device=cuda, dtype=torch.int32), torch.from_numpy(np.diff(indptr)).to(cuda))
        seeds_h = np.random.default_rng(3).permutation(n)[:1024].astype(np.int32)
        seeds = torch.from_numpy(seeds_h).to(cuda)
        fanouts = [15, 10, 5]
        ext.manual_seed(21)
        input_nodes, output_nodes, blocks = reference_layer_loop(ext, edge_src, edge_dst, edge_ptr, n, seeds, fanouts)
        # the oracle's loop draws hop h from stream h, as the module's per-call counter does after manual_seed
        w_inp, w_blocks = oracle.sample_blocks(indptr.astype(ptr_dtype), indices, seeds_h, fanouts, 21, 0)
        assert torch.equal(output_nodes, seeds)
        assert np.array_equal(input_nodes.cpu().numpy(), w_inp)
        for (src, dst, n_src, n_dst, src_g), w in zip(blocks, w_blocks):
            assert (n_src, n_dst) == (w["n_src"], w["n_dst"])
            assert np.array_equal(src.cpu().numpy(), w["src_local"])
            assert np.array_equal(src_g.cpu().numpy(), w["src_global"])
            assert np.array_equal(dst.cpu().numpy(), np.repeat(np.arange(n_dst), np.diff(w["indptr"])))

    # one GCN layer and one GIN layer on the outermost block, as GraphConv.py drives them
    src, dst, n_src, n_dst, _ = blocks[0]
    w0 = w_blocks[0]
    raw_dst_norm_degs = ext.cal_deg(dst.int(), n_dst)
    edge_ptr_b = ext.exclusive_sum(raw_dst_norm_degs)
    assert np.array_equal(edge_ptr_b.cpu().numpy(), w0["indptr"])
    src_norm_degs = ext.cal_deg(src.int(), n_src).clamp(min=1)
    dst_norm_degs = raw_dst_norm_degs.clamp(min=1)
    sn_h, dn_h = src_norm_degs.cpu().numpy(), dst_norm_degs.cpu().numpy()
    rng = np.random.default_rng(8)
    X = torch.from_numpy(rng.standard_normal((n_src, 32)).astype(np.float32)).to(cuda)
    W = torch.from_numpy(rng.standard_normal((32, 16)).astype(np.float32)).to(cuda)
    d_out = torch.from_numpy(rng.standard_normal((n_dst, 16)).astype(np.float32)).to(cuda)
    on_gpu = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(cuda)
    ptr_h, src_h = w0["indptr"], w0["src_local"]
    t_ptr, t_idx = oracle.transpose(ptr_h, src_h, n_src)
    # (products formed with the same library call on both sides: what is compared is the aggregation, at 1e-5)
    (out,) = ext.forward_gcn(edge_ptr_b, src.int(), src_norm_degs, dst_norm_degs, X, W, fanouts[0], n_dst)
    assert rel_err(out, oracle.aggregate(ptr_h, src_h, torch.mm(X, W).cpu().numpy(), "gcn", 0, dn_h, sn_h)) <= 1e-5
    d_x, d_w = ext.backward_gcn(edge_ptr_b, src.int(), dst_norm_degs, src_norm_degs, d_out, W, X)  # (dst, src): GraphConv.py:37
    G = oracle.aggregate(t_ptr, t_idx, d_out.cpu().numpy(), "gcn", 1, sn_h, dn_h)
    assert rel_err(d_x, torch.mm(on_gpu(G), W.t()).cpu().numpy()) <= 1e-5
    assert rel_err(d_w, torch.mm(X.t(), on_gpu(G)).cpu().numpy()) <= 1e-5
    out, tmp = ext.forwaed_gin(edge_ptr_b, src.int(), X, W, fanouts[0], n_dst)
    want_tmp = oracle.aggregate(ptr_h, src_h, X.cpu().numpy(), "sum", 0)
    assert rel_err(tmp, want_tmp) <= 1e-5
    assert rel_err(out, torch.mm(on_gpu(want_tmp), W).cpu().numpy()) <= 1e-5
    d_x, d_w = ext.backward_gin(edge_ptr_b, src.int(), d_out, W, tmp, n_src)
    assert rel_err(d_x, oracle.aggregate(t_ptr, t_idx, torch.mm(d_out, W.t()).cpu().numpy(), "sum", 1)) <= 1e-5
    assert rel_err(d_w, torch.mm(on_gpu(want_tmp).t(), d_out).cpu().numpy()) <= 1e-5
    # GAT aggregation with per-edge, per-head weights
    H = 4
    alpha = torch.from_numpy(rng.random((src.numel(), H, 1)).astype(np.float32)).to(cuda)
    (xg,) = ext.forward_gat(edge_ptr_b, alpha, src.int(), X, fanouts[0], n_dst, H)
    assert rel_err(xg, oracle.aggregate_edge(ptr_h, src_h, X.cpu().numpy(), alpha.view(-1, H).cpu().numpy(), zero_policy=0)) <= 1e-5
    (dxg,) = ext.backward_gat(edge_ptr_b, alpha, src.int(), d_out, n_src, H)
    tp, ti, te = oracle.transpose_with_edges(ptr_h, src_h, n_src)
    assert rel_err(dxg, oracle.aggregate_edge(tp, ti, d_out.cpu().numpy(), alpha.view(-1, H).cpu().numpy(), 1, edge_index=te)) <= 1e-5


def test_compiled_module_errors_are_runtime_errors(cuda, ext):
    cpu = torch.zeros(4, dtype=torch.int32)
    with pytest.raises(RuntimeError, match="CUDA tensor"):
        ext.cal_deg(cpu, 4)
    d = torch.zeros(8, dtype=torch.int32, device=cuda)
    with pytest.raises(RuntimeError, match="contiguous"):
        ext.cal_deg(d[::2], 4)
    with pytest.raises(RuntimeError, match="int32"):
        ext.exclusive_sum(d.long())
    ptr = torch.tensor([0, 2, 4], dtype=torch.int32, device=cuda)
    idx = torch.tensor([1, 0, 0, 1], dtype=torch.int32, device=cuda)
    with pytest.raises(RuntimeError, match="outside the graph"):
        ext.sample_node(idx, idx, ptr, torch.tensor([0, 5], dtype=torch.int32, device=cuda), 2, 2)
    with pytest.raises(RuntimeError, match="negative id"):
        ext.transfer_edge_id(torch.tensor([1, -1], dtype=torch.int32, device=cuda), torch.tensor([0, 0], dtype=torch.int32, device=cuda),
                             torch.tensor([0], dtype=torch.int32, device=cuda), 1, 3, 2, 2)


def test_weight_gradients_follow_grad_mode_and_autocast(ext, cuda):
    """The dense products of backward_gin are torch's where a graph is being recorded or autocast picks the types."""
    import fastgl
    ptr = torch.arange(0, 41, 4, dtype=torch.int32, device=cuda)
    src = torch.arange(40, dtype=torch.int32, device=cuda) % 20
    d, w, x = (torch.randn(s, device=cuda) for s in ((10, 8), (6, 8), (10, 6)))
    want = x.t() @ d
    _, d_w = ext.backward_gin(ptr, src, d, w, x, 20)
    assert rel_err(d_w, want.cpu().numpy()) < 1e-5 and not d_w.requires_grad
    _, d_w = ext.backward_gin(ptr, src, d, w, x.clone().requires_grad_(True), 20)
    assert d_w.requires_grad and rel_err(d_w.detach(), want.cpu().numpy()) < 1e-5
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert fastgl.ops.weight_grad(x, d).dtype == torch.bfloat16


@pytest.mark.parametrize("stride", [1, 1 << 24])
def test_weight_gradient_of_a_single_row(ext, cuda, stride):
    """A single row is contiguous whatever its row stride says."""
    ptr = torch.tensor([0, 1], dtype=torch.int32, device=cuda)
    idx = torch.zeros(1, dtype=torch.int32, device=cuda)
    x, g, w = (torch.randn(s, device=cuda) for s in (20, 7, (20, 7)))
    x, g = x.as_strided((1, 20), (stride, 1)), g.as_strided((1, 7), (stride, 1))
    assert x.is_contiguous() and g.is_contiguous()
    one = torch.ones(1, dtype=torch.int32, device=cuda)
    for d_x, d_w in (ext.backward_gin(ptr, idx, g, w, x, 1), ext.backward_gcn(ptr, idx, one, one, torch.cat([g[0]]).view(1, 7), w, x)):
        assert torch.allclose(d_w, x.t() @ g, rtol=1e-5, atol=1e-5) and torch.allclose(d_x, g @ w.t(), rtol=1e-5, atol=1e-5)


def test_dispatch_modes_see_the_weight_gradient(ext, cuda):
    from torch.utils.flop_counter import FlopCounterMode
    ptr = torch.arange(6, dtype=torch.int32, device=cuda)
    idx = torch.arange(5, dtype=torch.int32, device=cuda)
    x, g, w = (torch.randn(s, device=cuda) for s in ((5, 20), (5, 7), (20, 7)))
    with FlopCounterMode(display=False) as count:
        ext.backward_gin(ptr, idx, g, w, x, 5)
    assert count.get_total_flops() == 2 * 2 * 5 * 20 * 7  # the input's gradient and the weight's
