"""Rows of a sorted transposed block around the sizes at which the sort takes them apart -- a wave's 64 entries, pieces of 2048 -- against
the oracle's stable transpose, through a batch whose seeds all have one neighbour, so that a hub's row has exactly the length that is asked for."""
import numpy as np
import pytest

from test_gpu_idmap_blocks import _csr_from_rows, dev_i32, load_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [(64, 65, 128, 129), (2047, 2048, 2049), (4095, 4096, 4097, 1), (6144, 6145), (40_000, 3, 2050, 66)])
def test_rows_of_these_lengths(cuda, oracle, lengths):
    import fastgl
    print("sorted pieces", lengths, flush=True)
    rng = np.random.default_rng(sum(lengths))
    n_seeds = sum(lengths)
    target = n_seeds + np.repeat(np.arange(len(lengths)), lengths)
    rng.shuffle(target)
    rows = [[int(t)] for t in target] + [[] for _ in lengths]
    indptr, indices = _csr_from_rows(rows)
    ptr, idx = load_graph(cuda, indptr, indices)
    seeds = rng.permutation(n_seeds).astype(np.int32)
    sampler = fastgl.FusedMapSampler([2], rng_seed=1, deterministic=True, transposed="all").set_graph(ptr, idx)
    for it in range(2):
        _, _, (b,) = sampler.sample_blocks(None, dev_i32(seeds, cuda))
        _, (w,) = oracle.sample_blocks(indptr, indices, seeds, [2], 1, 64 * it)
        t_ptr, t_dst, t_edge = (t.cpu().numpy() for t in b.transposed(edge_ids=True))
        w_ptr, w_idx = oracle.transpose(w["indptr"], w["src_local"], w["n_src"])
        assert np.array_equal(t_ptr, w_ptr) and np.array_equal(t_dst, w_idx)
        assert sorted(np.diff(w_ptr).tolist())[-len(lengths):] == sorted(lengths)
        assert np.array_equal(t_edge, np.argsort(w["src_local"], kind="stable"))
