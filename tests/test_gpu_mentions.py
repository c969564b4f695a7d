"""First mentions of new ids, marked while they are being inserted: the sizes at which the number pass changes the way it counts
the marks, hops that insert while they sample and hops that do not, and hops that outgrow the unique list, against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev_i32(a, cuda):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).to(cuda)


# 512 edges: a line of marks; 4096: a tile of lines; 2048 x 512: the last size whose marks every workgroup counts itself;
# 2048 x 4096: the last whose tiles every workgroup scans itself
@pytest.mark.parametrize("n_edges", [1, 63, 64, 65, 511, 512, 513, 4095, 4096, 4097, 2048 * 512, 2048 * 512 + 1, 2048 * 4096, 2048 * 4096 + 1])
@pytest.mark.parametrize("order", ["ascending", "descending", "shuffled"])
def test_numbering_at_the_edges_of_lines_and_tiles(cuda, oracle, n_edges, order):
    import fastgl
    print("mentions %d %s" % (n_edges, order), flush=True)
    if n_edges > 4097 and order != "shuffled":
        pytest.skip("the large sizes once")
    rng = np.random.default_rng(n_edges)
    n_dst = min(n_edges, 300)
    dst_unique = rng.choice(10_000, size=n_dst, replace=False).astype(np.int32)
    # every id twice: in ascending, descending or any order, so that first mentions are displaced in every line
    src = (np.arange(n_edges, dtype=np.int64) // 2 * 3 + 20_000).astype(np.int32)
    src = {"ascending": src, "descending": src[::-1].copy(), "shuffled": rng.permutation(src)}[order]
    src[::5] = dst_unique[rng.integers(0, n_dst, size=src[::5].size)]
    dst = dst_unique[np.sort(rng.integers(0, n_dst, size=n_edges))]
    w_src, w_dst, w_uniq = oracle.idmap(src, dst, dst_unique)
    got = fastgl.transfer_edge_id(dev_i32(src, cuda), dev_i32(dst, cuda), dev_i32(dst_unique, cuda), n_dst, n_dst + n_edges, 1 << 30, n_edges)
    assert np.array_equal(got[0].cpu().numpy(), w_src) and np.array_equal(got[1].cpu().numpy(), w_dst)
    assert np.array_equal(got[2].cpu().numpy(), w_uniq)


# hops of up to 262144 seeds (in the plan's bounds) and fanout 32 insert while they sample, 16 seeds a workgroup and 64 to an entry of the tile
# sums; fanouts beyond 32 do not, with 64 seeds a tile, nor do larger hops, with 256 (64 beyond fanout 48).  120000 seeds: the second hop's tiles are
# others than the first's
@pytest.mark.parametrize("n_seeds,fanouts", [(1, [3, 2]), (15, [5, 8]), (16, [9, 8]), (17, [9, 8]), (64, [8, 9]), (65, [16, 17]), (63, [32, 1]), (640, [33, 5]),
                                             (65_536, [4]), (65_537, [4]), (262_144, [4]), (262_145, [4]), (120_000, [2, 4]), (120_000, [33, 4]),
                                             (120_000, [49, 4]), (100, [6, 6, 6, 6])])
@pytest.mark.parametrize("transposed", ["none", "inner", "all"])
def test_hops_on_both_sides_of_the_line(cuda, oracle, n_seeds, fanouts, transposed):
    import fastgl
    print("hops %d %s %s" % (n_seeds, fanouts, transposed), flush=True)
    n_nodes = 70_000 if n_seeds <= 65_537 else 300_000
    indptr, indices = oracle.rmat_csr(n_nodes, 10 * n_nodes, seed=3)
    seeds = np.random.default_rng(n_seeds).permutation(n_nodes)[:n_seeds].astype(np.int32)
    sampler = fastgl.FusedMapSampler(fanouts, rng_seed=5, deterministic=True, transposed=transposed).set_graph(
        torch.from_numpy(indptr).to(cuda), torch.from_numpy(indices).to(cuda))
    for it in range(3):
        inp, _, blocks = sampler.sample_blocks(None, dev_i32(seeds, cuda))
        w_inp, w_blocks = oracle.sample_blocks(indptr, indices, seeds, fanouts, 5, it * 64)
        assert np.array_equal(inp.cpu().numpy(), w_inp)
        for b, w in zip(blocks, w_blocks):
            assert np.array_equal(b.edge_ptr.cpu().numpy(), w["indptr"]) and np.array_equal(b.src_local.cpu().numpy(), w["src_local"])
            want = oracle.transpose(w["indptr"], w["src_local"], w["n_src"])
            got = [t.cpu().numpy() for t in b.transposed()]
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("caps", [[256, 256, 256, 256, 256], [256, 300, 310, 900, 5000], [256, 700, 701, 701, 702]])
def test_hops_that_outgrow_the_unique_list_leave_no_position_unwritten(cuda, oracle, caps):
    """An id that found no room stays unnumbered in the table; the hops behind must not take its edge for one of theirs: every
    position up to the clamped node count holds a node, whatever the workspace held before."""
    import fastgl
    print("overflow %s" % caps, flush=True)
    indptr, indices = oracle.rmat_csr(20_000, 200_000, seed=1)
    ptr, idx = torch.from_numpy(indptr).to(cuda), torch.from_numpy(indices).to(cuda)
    hubs = np.argsort(-np.diff(indptr))[:256].astype(np.int32)
    plan = fastgl.BlocksPlan(indptr.size - 1, 256, [5, 10, 15, 10], cuda, node_capacity=caps, transpose_hops=(0, 1, 2))
    for it in range(4):
        plan.ws.fill_(0)
        out = fastgl.sample_blocks_fused(plan, ptr, idx, dev_i32(hubs, cuda), 9, 64 * it)
        c = out[4].tolist()
        assert c[2 * 4 + 1] & 2  # FGL_STATUS_UNIQ_OVERFLOW
        assert all(a <= b for a, b in zip(c[:5], caps))
        uniq = out[0][:c[4]].cpu().numpy()
        assert np.array_equal(uniq[:256], hubs) and uniq.min() >= 0 and uniq.max() < 20_000 and np.unique(uniq).size == uniq.size
        for h in range(4):
            e_ptr = out[1][h][:c[h] + 1].cpu().numpy()
            want = np.minimum(np.diff(indptr)[uniq[:c[h]]], [5, 10, 15, 10][h])
            assert np.array_equal(np.diff(e_ptr), want)
