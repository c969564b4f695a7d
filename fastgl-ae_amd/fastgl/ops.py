"""The operator functions of the reference's ``fastgl`` extension module, with the same
names, positional arguments, return lists and error type (cuda_operators/aggregate_acc.cpp:
601-621 lists them; only the ones its Python code calls are provided), implemented over
the HIP C ABI.  Extensions that the reference does not have (mean aggregation, the
transposed block, the all-hops sampler) follow at the end.

Index tensors are int32 and must be contiguous device tensors (``RuntimeError`` otherwise,
as the reference's CHECK_INPUT, aggregate_acc.cpp:4-6); ``edge_ptr`` of the full graph may
also be int64.  Features are fp32 or bf16.
"""
from __future__ import annotations

import ctypes as C

import torch
from torch.utils._device import DeviceContext

from . import _lib as L

_rng_state = {"seed": 0, "calls": 0}


def manual_seed(seed: int) -> None:
    """Seed of the sampler's Philox streams; also resets the per-call stream counter.
    (The reference's picks come from one constant stream, sample.cu:70.)"""
    _rng_state["seed"] = int(seed) & 0xFFFFFFFFFFFFFFFF
    _rng_state["calls"] = 0


def _check_input(t, name, dtypes=None):
    if not isinstance(t, torch.Tensor):
        raise RuntimeError("%s must be a tensor" % name)
    if not t.is_cuda:
        raise RuntimeError("%s must be a CUDA tensor" % name)
    if not t.is_contiguous():
        raise RuntimeError("%s must be contiguous" % name)
    if dtypes is not None and t.dtype not in dtypes:
        raise RuntimeError("%s must have dtype in %s, got %s" % (name, [str(d) for d in dtypes], t.dtype))


class _NoSwitch:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_NO_SWITCH = _NoSwitch()


def _on_device(dev):
    """Context that makes ``dev`` the current device -- nothing at all when it already is (the usual case: entering
    and leaving ``torch.cuda.device`` costs several microseconds per call)."""
    index = dev.index
    if index is None or index == torch.cuda.current_device():
        return _NO_SWITCH
    return torch.cuda.device(dev)


def _same_device(*tensors):
    dev = tensors[0].device
    for t in tensors[1:]:
        if t is not None and t.device != dev:
            raise RuntimeError("all tensors must live on the same device")
    return dev


_I32 = (torch.int32,)
_PTR = (torch.int32, torch.int64)
_FEAT = (torch.float32, torch.bfloat16)


def _raise_status(bits: int, where: str):
    if bits:
        raise RuntimeError("fastgl.%s: %s" % (where, L.status_message(bits)))


# ---------------------------------------------------------------------------------------
# drop-in operators
# ---------------------------------------------------------------------------------------
_host_words = {}


def _expect_sizes(dev, stream):
    """Two pinned host words per (device, stream) for a call's ``{size, status}``, marked pending: the call's kernels
    store both there themselves (no copy to enqueue), ``_sizes`` waits for them."""
    key = (torch.device(dev).index, stream)
    h = _host_words.get(key)
    if h is None:
        h = _host_words[key] = torch.empty(2, dtype=torch.int32, pin_memory=True)
    h.fill_(-1)  # (no size and no status word is all ones)
    return h


def _sizes(h, stream):
    L.check(L.lib().fgl_wait_words(h.data_ptr(), 2, -1, stream, 5000))
    return h.tolist()


def sample_node(src_edges, dst_edges, edge_ptr, seed_nodes, dst_nodes, neighbor_num):
    """fastgl.sample_node (aggregate_acc.cpp:491-512): ``-> [src_out, dst_out, edges_num]``.

    ``src_edges`` is the CSR ``indices`` of the in-neighbour graph, ``edge_ptr`` its
    ``indptr``; ``dst_edges`` is accepted and, as in the reference kernels, never read.
    Outputs hold global ids, each seed's edges contiguous, seeds in order.
    """
    _check_input(src_edges, "src_edges", _I32)
    _check_input(dst_edges, "dst_edges")
    _check_input(edge_ptr, "edge_ptr", _PTR)
    _check_input(seed_nodes, "seed_nodes", _I32)
    dev = _same_device(src_edges, edge_ptr, seed_nodes)
    n_seeds = int(seed_nodes.size(0))
    dst_nodes = int(dst_nodes)
    fanout = int(neighbor_num)
    if dst_nodes < n_seeds:
        raise RuntimeError("dst_nodes (%d) is smaller than the number of seeds (%d)" % (dst_nodes, n_seeds))
    lib = L.lib()
    with _on_device(dev):
        src_out = torch.empty(max(dst_nodes * fanout, 1), dtype=torch.int32, device=dev)
        dst_out = torch.empty(max(dst_nodes * fanout, 1), dtype=torch.int32, device=dev)
        block_ptr = torch.empty(n_seeds + 1, dtype=torch.int32, device=dev)
        meta = torch.zeros(2, dtype=torch.int32, device=dev)  # [edge count, status]
        ws_bytes = lib.fgl_sample_workspace_bytes(n_seeds, fanout)
        ws = L.workspace(ws_bytes, dev)
        stream_id = _rng_state["calls"] & 0xFFFFFFFF
        _rng_state["calls"] += 1
        st = L.stream_handle()
        host = _expect_sizes(dev, st)
        L.check(lib.fgl_sample_node(L.ptr(edge_ptr), int(edge_ptr.dtype == torch.int64), L.ptr(src_edges),
                                    int(edge_ptr.size(0)) - 1, L.ptr(seed_nodes), n_seeds, None, fanout,
                                    _rng_state["seed"], stream_id, L.ptr(src_out), L.ptr(dst_out), L.ptr(block_ptr),
                                    meta.data_ptr(), meta.data_ptr() + 4, host.data_ptr(), L.ptr(ws), ws.numel(), st))
        n_edges, status = _sizes(host, st)  # the host read-back the reference also does (sample.cu:202)
    _raise_status(status, "sample_node")
    edges_num = meta[:1]
    out = [src_out[:n_edges], dst_out[:n_edges], edges_num]
    sample_node.last_block_ptr = block_ptr  # CSR offsets of the block just sampled
    return out


sample_node.last_block_ptr = None


def transfer_edge_id(src_edges, dst_edges, dst_edges_unique, dst_nodes, total_items, unique_num, edge_nums):
    """fastgl.transfer_edge_id (aggregate_acc.cpp:467-489, id_map.cu:386-493): the fused
    id-map.  Rewrites ``src_edges`` / ``dst_edges`` in place to local ids and returns
    ``[src_edges, dst_edges, uniq]`` with ``uniq = cat(dst_edges_unique, new source ids)``.
    New ids are numbered in first-occurrence order."""
    _check_input(src_edges, "src_edges", _I32)
    _check_input(dst_edges, "dst_edges", _I32)
    _check_input(dst_edges_unique, "dst_edges_unique", _I32)
    dev = _same_device(src_edges, dst_edges, dst_edges_unique)
    n_dst = int(dst_nodes)
    n_edges = int(edge_nums)
    if n_dst > dst_edges_unique.size(0):
        raise RuntimeError("dst_nodes (%d) exceeds len(dst_edges_unique) (%d)" % (n_dst, dst_edges_unique.size(0)))
    if n_edges > src_edges.size(0) or n_edges > dst_edges.size(0):
        raise RuntimeError("edge_nums (%d) exceeds the edge arrays" % n_edges)
    if int(total_items) - n_dst != n_edges:
        raise RuntimeError("total_items - dst_nodes must equal edge_nums (id_map.cu:308)")
    lib = L.lib()
    max_new = max(0, min(int(unique_num), n_edges))
    capacity = n_dst + max_new
    slots = lib.fgl_idmap_slots(capacity)
    with _on_device(dev):
        st = L.stream_handle()
        key = (torch.device(dev).index, st)
        table, known_empty = _table(slots, dev)
        uniq = torch.empty(max(capacity, 1), dtype=torch.int32, device=dev)
        meta = torch.zeros(2, dtype=torch.int32, device=dev)  # [n_total, status]
        ws_bytes = lib.fgl_idmap_map_src_workspace_bytes(n_edges)
        ws = L.workspace(ws_bytes, dev)
        status_ptr = meta.data_ptr() + 4
        # the table is a prefix of a persistent buffer that every call leaves empty: only slots that no call has
        # emptied yet are filled here (in the steady state of a training loop: none)
        if known_empty < slots:
            L.check(lib.fgl_idmap_reset(L.ptr(table), slots, st))
        _tables[key] = (table, 0)
        host = _expect_sizes(dev, st)
        # destination ids in, then three passes over the edges (the destination half rides on the first); the last
        # writes nothing back into the table (no later call looks these ids up) and empties it
        L.check(lib.fgl_idmap_transfer(L.ptr(table), slots, L.ptr(dst_edges_unique), n_dst, L.ptr(src_edges), L.ptr(dst_edges),
                                       n_edges, L.ptr(uniq), capacity,
                                       L.IDMAP_ORDERED | L.IDMAP_FINAL | L.IDMAP_LEAVE_TABLE_EMPTY, meta.data_ptr(), status_ptr,
                                       host.data_ptr(), L.ptr(ws), ws.numel(), st))
        _tables[key] = (table, max(known_empty, slots))
        n_total, status = _sizes(host, st)  # host read-back, as id_map.cu:454,491
    _raise_status(status, "transfer_edge_id")
    return [src_edges, dst_edges, uniq[:n_total]]


_tables = {}


def _table(slots: int, dev):
    """Hash-table storage, cached per (device, stream) and grown on demand (the reference
    cudaMallocs, memsets and cudaFrees one per call, id_map.cu:45-59), with the number of its leading slots
    that are known to hold the empty marker."""
    key = (torch.device(dev).index, L.stream_handle())
    t, known_empty = _tables.get(key, (None, 0))
    if t is None or t.numel() < slots:
        t, known_empty = torch.empty(int(slots), dtype=torch.int64, device=dev), 0
        _tables[key] = (t, 0)
    return t, known_empty


def cal_deg(edges, nodes_num):
    """fastgl.cal_deg (aggregate_acc.cpp:522-529): int32 histogram of ``edges`` over ``nodes_num`` bins."""
    _check_input(edges, "edges", _I32)
    n = int(nodes_num)
    dev = edges.device
    with _on_device(dev):
        deg = torch.empty(max(n, 1), dtype=torch.int32, device=dev)[:n]
        lib = L.lib()
        ws_bytes = lib.fgl_cal_deg_workspace_bytes(int(edges.numel()), n)
        ws = L.workspace(ws_bytes, dev) if ws_bytes else None
        L.check(lib.fgl_cal_deg_ws(L.ptr(edges), int(edges.numel()), None, L.ptr(deg), n, L.ptr(ws), ws_bytes, L.stream_handle()))
    return deg


def exclusive_sum(in_degs):
    """fastgl.exclusive_sum (aggregate_acc.cpp:514-520): ``len+1`` exclusive prefix sums (int32)."""
    _check_input(in_degs, "in_degs", _I32)
    n = int(in_degs.numel())
    dev = in_degs.device
    lib = L.lib()
    with _on_device(dev):
        out = torch.empty(n + 1, dtype=torch.int32, device=dev)
        ws = L.workspace(lib.fgl_exclusive_sum_workspace_bytes(n), dev)
        L.check(lib.fgl_exclusive_sum_i32(L.ptr(in_degs), n, None, L.ptr(out), L.ptr(ws), ws.numel(), L.stream_handle()))
    return out


def _fanout_bound(edge_ptr, neighbor_num):
    """``neighbor_num`` bounds the entries per row of a sampled block (the reference sizes its shared
    staging by it, aggregate_acc_kernel.cu:238-247)."""
    bound = getattr(edge_ptr, "fgl_longest_row", None)
    if bound is None and int(neighbor_num) > 0:
        bound = int(neighbor_num)
    return bound


def forward_gcn(edge_ptr, src_edges, src_norm_degs, dst_norm_degs, input_feat, weight, neighbor_num, dst_nodes):
    """fastgl.forward_gcn (aggregate_acc.cpp:133-160): ``[A_norm (X W)]`` with
    ``A_norm[d, s] = 1/sqrt(dst_norm[d]) * 1/sqrt(src_norm[s])``; a dst row without edges
    passes ``(X W)[d]`` through (aggregate_acc_kernel.cu:307-309)."""
    for t, n in ((edge_ptr, "edge_ptr"), (src_edges, "src_edges"), (src_norm_degs, "src_norm_degs"),
                 (dst_norm_degs, "dst_norm_degs")):
        _check_input(t, n, _I32)
    _check_input(input_feat, "input_feat", _FEAT)
    _check_input(weight, "weight", _FEAT)
    tmp = row_product(input_feat, weight)
    out = aggregate(edge_ptr, src_edges, tmp, mode="gcn", zero_policy="self", row_norm=dst_norm_degs,
                    col_norm=src_norm_degs, n_rows=int(dst_nodes), longest_row=_fanout_bound(edge_ptr, neighbor_num))
    return [out]


def backward_gcn(edge_ptr, src_edges, src_norm_degs, dst_norm_degs, d_input, weight, input_feat):
    """fastgl.backward_gcn (aggregate_acc.cpp:349-376): ``[d_x, d_w]``.

    Positional meaning as in the reference kernel (aggregate_acc_kernel.cu:494,509): the
    third argument is indexed by destination id and the fourth by source id -- the caller
    passes ``(dst_norm, src_norm)`` there (GraphConv.py:37)."""
    by_dst, by_src = src_norm_degs, dst_norm_degs
    for t, n in ((edge_ptr, "edge_ptr"), (src_edges, "src_edges"), (by_dst, "src_norm_degs"), (by_src, "dst_norm_degs")):
        _check_input(t, n, _I32)
    _check_input(d_input, "d_input", _FEAT)
    _check_input(weight, "weight", _FEAT)
    _check_input(input_feat, "input_feat", _FEAT)
    n_src = int(input_feat.size(0))
    n_dst = int(d_input.size(0))
    t_ptr, t_idx = block_transpose(edge_ptr, src_edges, n_dst, n_src)
    g = aggregate(t_ptr, t_idx, d_input, mode="gcn", zero_policy="zeros", row_norm=by_src, col_norm=by_dst, n_rows=n_src)
    d_x = row_product(g, weight, transposed=True)
    d_w = weight_grad(input_feat, g)
    return [d_x, d_w]


def forwaed_gin(edge_ptr, src_edges, input_feat, weight, neighbor_num, dst_nodes):
    """fastgl.forwaed_gin (sic; aggregate_acc.cpp:173-199, exported at :613): ``[tmp W, tmp]``
    with ``tmp[d] = sum of X[s] over the edges into d`` (``X[d]`` if there are none)."""
    _check_input(edge_ptr, "edge_ptr", _I32)
    _check_input(src_edges, "src_edges", _I32)
    _check_input(input_feat, "input_feat", _FEAT)
    _check_input(weight, "weight", _FEAT)
    tmp = aggregate(edge_ptr, src_edges, input_feat, mode="sum", zero_policy="self", n_rows=int(dst_nodes),
                    longest_row=_fanout_bound(edge_ptr, neighbor_num))
    return [row_product(tmp, weight), tmp]


def backward_gin(edge_ptr, src_edges, d_input, weight, input_feat, src_nodes):
    """fastgl.backward_gin (aggregate_acc.cpp:387-409): ``[d_x, d_w]``; ``input_feat`` is the
    ``tmp`` that forwaed_gin returned."""
    _check_input(edge_ptr, "edge_ptr", _I32)
    _check_input(src_edges, "src_edges", _I32)
    _check_input(d_input, "d_input", _FEAT)
    _check_input(weight, "weight", _FEAT)
    _check_input(input_feat, "input_feat", _FEAT)
    d_tmp = row_product(d_input, weight, transposed=True)
    d_w = weight_grad(input_feat, d_input)
    n_dst = int(d_input.size(0))
    t_ptr, t_idx = block_transpose(edge_ptr, src_edges, n_dst, int(src_nodes))
    d_x = aggregate(t_ptr, t_idx, d_tmp, mode="sum", zero_policy="zeros", n_rows=int(src_nodes))
    return [d_x, d_w]


def forward_gat(edge_ptr, edge_data, src_edges, input_feat, neighbor_num, dst_nodes, num_heads):
    """fastgl.forward_gat (aggregate_acc.cpp, kernel aggregate_acc_kernel.cu:835-886):
    ``[out]`` with ``out[d, f] = sum_e edge_data[e, f // (D / num_heads)] * input_feat[src[e], f]``
    (``input_feat[d]`` if d has no edges)."""
    _check_input(edge_ptr, "edge_ptr", _I32)
    _check_input(src_edges, "src_edges", _I32)
    _check_input(edge_data, "edge_data", (torch.float32,))
    _check_input(input_feat, "input_feat", _FEAT)
    return [aggregate(edge_ptr, src_edges, input_feat, mode="edge", zero_policy="self", n_rows=int(dst_nodes),
                      edge_weight=edge_data.view(edge_data.size(0), -1), n_heads=int(num_heads))]


def backward_gat(edge_ptr, edge_data, src_edges, d_input, src_nodes, num_heads):
    """fastgl.backward_gat (kernel aggregate_acc_kernel.cu:924-979): ``[d_x]`` with
    ``d_x[s, f] = sum over the edges (s -> d) of edge_data[e, head(f)] * d_input[d, f]`` -- as a gather
    over the transposed block instead of float atomics."""
    _check_input(edge_ptr, "edge_ptr", _I32)
    _check_input(src_edges, "src_edges", _I32)
    _check_input(edge_data, "edge_data", (torch.float32,))
    _check_input(d_input, "d_input", _FEAT)
    n_dst = int(d_input.size(0))
    t_ptr, t_idx, t_edge = block_transpose(edge_ptr, src_edges, n_dst, int(src_nodes), edge_ids=True)
    return [aggregate(t_ptr, t_idx, d_input, mode="edge", zero_policy="zeros", n_rows=int(src_nodes),
                      edge_weight=edge_data.view(edge_data.size(0), -1), n_heads=int(num_heads), edge_index=t_edge)]


# ---------------------------------------------------------------------------------------
# extensions
# ---------------------------------------------------------------------------------------
_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
_transforms = torch._C._functorch.peek_interpreter_stack


def _followed():
    """Whether something follows torch's operators as they are called and would miss a product that does not go through one: a
    transform of ``torch.func``, a tracer, a FLOP counter or another dispatch or function mode.  (A default device is a function mode
    too, and follows nothing.)"""
    if _dispatch_modes() > 0 or _transforms() is not None:
        return True
    n = _function_modes()
    return n > 0 and any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(n))


def _addresses(a, b):
    """Where the two tensors lie, or None if one has no memory of its own: the gradients that ``torch.autograd.grad`` hands to
    backward passes with ``is_grads_batched`` (and ``jacobian`` with ``vectorize``) look like matrices, but only torch's operators take them."""
    try:
        return a.data_ptr(), b.data_ptr()
    except RuntimeError:
        return None


def _splits_k(k, m, n):
    """Whether ``weight_grad`` forms its product with the library's k-splitting kernel.  A weight gradient has a few output
    tiles and a long k, where a GEMM that parallelises over tiles leaves the chip idle (100 x 256 outputs, k = 105 K: fp32
    190 -> 72 us, bf16 245 -> 25 us; 256 x 256, k = 500: 119 -> 27 us).  Many tiles and a short k are the library GEMM's
    (1024 x 1024, k = 8192: 145 us against 268 in fp32, 57 against 63 in bf16; 256 x 1024, k = 2000: 20 against 31)."""
    return m * n <= 65536 or k * k >= 256 * m * n


def _long_product_is_the_kernels(dtype, transposed, k, n):
    """Beyond 8e9 multiplications: whether the kernel is ahead of the library for a product of k x n.  A short k leaves little to multiply for each
    row that moves, and the library moves rows at half the memory's rate: up to k = 32 in fp32, and in bf16 up to 128 (transposed: 100), the kernel is
    ahead.  For a longer k in fp32 it depends on what either pads.  The library is slow where a row is no whole number of 64-byte lines (a
    sixteenth of the sizes is its own, then); the kernel works in 32 columns a wave, one vector of two or four a lane where that pads little, so
    that 65 .. 80 columns cost it as much as 96, one by one, and 129 .. 160 as much as 192.  The lines lie where sweeps of n = 33 .. 330 cross, k = 36 .. 128.
    Kernel's time over the library's, 9e9 multiplications (transposed), k = 64 / 100 / 128: 40 columns 0.96 / 1.01 / 1.19 (0.61 / 0.62 / 0.69), 50 columns
    0.78 / 0.76 / 0.94 (0.85 / 0.87 / 1.01), 72 columns 1.06 / 1.44 / 1.48 (1.13 / 0.79 / 0.86), 80 columns 1.38 / 1.50 / - (1.49 / 1.66 / -), 90 columns 0.87 /
    0.95 / 1.01 (0.93 / 1.11 / 1.18), 100 columns 0.62 / 0.87 / 0.82 (0.70 / 0.47 / 0.88), 120 columns 0.58 / 0.76 / 0.82 (0.66 / 0.91 / 0.89), 130 columns 1.21 /
    1.35 / 1.29 (1.09 / 0.56 / 0.62), 250 columns 0.47 / 0.82 / 0.51 (0.68 / 0.81 / 0.86), 300 columns 0.66 / 0.89 / 0.98 (0.72 / 0.84 / 1.08); 128 x 64 is
    the library's in both layouts.  bf16, k = 64 / 100 / 128: 64 columns 0.61 / 0.62 / 0.86, 100 columns 0.30 / 0.36 / 0.43, but 96 columns, one by one again,
    0.78 / 0.86 / 1.09 and with k = 96 1.12 (1.19); transposed odd columns beyond 192, stored one by one, 0.83 / 1.06 / 1.33."""
    if dtype == torch.bfloat16:
        return k <= (100 if transposed else 128) and not (64 < n <= 96 and n % 16 == 0) and not (transposed and n > 192 and n % 2 == 1)
    if k <= 32:
        return True
    if k > 128 or n % 16 == 0:
        return False
    if n <= 192:
        return (32 if transposed else 48) < n < 64 or (96 if transposed else 80) < n < 128
    return k <= (100 if transposed else 128) and -(-n // 64) * 64 <= 1.15 * (-(-n // 16) * 16)


def _forms_row_product(a, b, transposed, m, k, n):
    """Whether ``row_product`` is the kernel's: plain matrices on one GPU of one type, nobody recording a graph of the call or following it,
    no autocast to change the types, and a size where steps over fresh blocks gain.  The library looks for a kernel on every call with sizes
    it has not just seen -- 74 us of the host's time against 12 -- which is what a product of a mini-batch takes.  On the GPU, sizes repeated (us,
    library / here): up to k = 128 the two are alike or this one is ahead (fp32 107 K x 100 x 256 81 / 78, 200 K x 128 x 128 81 / 85, 107 K x 64 x 64 29 / 21;
    bf16 29 / 24, 30 / 29, 22 / 8; with a transposed weight 84 / 84, 81 / 91, 29 / 20; bf16 30 / 30, 28 / 33, 20 / 10).  A longer k costs it more than the
    library, whose tiles go through LDS (256 x 256, fp32: 8192 rows 13 / 13, 20 K 26 / 43, 107 K 138 / 144, transposed 141 / 161; bf16: 7 / 7, 10 / 15, 28 / 39,
    transposed 27 / 52; 256 x 384 and 300 x 300 are no worse): a caller of ever the same sizes whom the GPU keeps waiting loses that much.  Steps
    over fresh blocks gain all the same: drawing the line for k > 128 at 2e9 instead made GCN inference of 256 x 256 (60 K rows) 330 -> 349 us, GraphSAGE in
    bf16, 87 K rows of 256 x 256, 996 -> 1294 us a training step and 360 -> 423 in inference, and 3 % better at most (in fp32, 1663 -> 1625).  Products beyond the
    line keep the GPU busy for longer than the host takes, and there it depends on the size (a GIN layer of 602 x 256 over 8192 rows, forward and backward, is the
    library's: 394 / 418 in all), see ``_long_product_is_the_kernels``.
    Returns the operands' addresses and row strides if so, else None."""
    if not (k * n <= 100000 and (m * k * n <= 8 * 10 ** 9 or _long_product_is_the_kernels(a.dtype, transposed, k, n))):
        return None
    return _product_operands(a, b, transposed, m, k, n)


def _product_operands(a, b, transposed, m, k, n):
    """The operands' addresses and row strides where fgl_row_product can take them, else None (see ``_forms_row_product``)."""
    if not (a.is_cuda and a.dtype == b.dtype and a.dtype in _FEAT and m > 0 and 0 < k <= 65536 and 0 < n <= 65536 and
            a.get_device() == b.get_device() and not (torch.is_grad_enabled() and (a.requires_grad or b.requires_grad)) and
            not torch.is_autocast_enabled() and not _followed()):
        return None
    (lda, unit_a), (ldb, unit_b), at = a.stride(), b.stride(), _addresses(a, b)
    if (at is not None and unit_a == 1 and lda >= k and unit_b == 1 and ldb >= b.size(1) and
            (a.dtype == torch.float32 or (lda % 2 == 0 and at[0] % 4 == 0 and (not transposed or (ldb % 2 == 0 and at[1] % 4 == 0))))):
        return at[0], lda, at[1], ldb
    return None


def _forms_split_product(a, b, transposed, m, k, n):
    """What ``_forms_row_product`` leaves, and the fp32 kernel on the bf16 matrix cores (csrc/fgl_split_product.hip) forms ahead of the
    library: more than 8e9 multiplications, or weights of more than 100000 values.  us, the library / that kernel, plain weight (T: transposed):
    2.4 M x 100 x 64 511 / 345, 2.4 M x 64 x 100 626 / 332, 1.2 M x 100 x 128 415 / 322; wide weights 8192 x 256 x 602 36 / 28 (T 33 / 28), 20 K
    rows 70 / 51 (69 / 52), 60 K 270 / 124 (218 / 126), 400 x 300: 8192 38 / 23, 60 K 179 / 99, 300 x 400: 8192 26 / 23; but 4000 rows of
    these two, fewer than 2.1e6 results, 18 / 22, and a k beyond 400, of which only 32 columns at a time fit, gains little or nothing: 602 x 256
    8192 rows 26.9 / 26.4, 20 K 53 / 60, 60 K 151 / 152, 107 K 320 / 300.  n = 66 to 71 in two workgroups' columns, n = 129 to 160 from
    k = 129 on and n of 33 to 48 from k = 257 on stay the library's too; that was ahead there by up to a fifth of misaligned stores and a last round
    with few workgroups, without which the kernel is (2.4 M x 100 x 66 655 / 556, 400 K x 200 x 160 330 / 240, 400 K x 400 x 47 204 / 178).
    From 4000 rows on, up to 30000 columns, 0.5 .. 0.83 of the library's time; fewer where they fill the XCDs' turns, 2048 rows each, 1024 up to
    k = 192 (2000 rows: k = 33 .. 400 0.6 .. 0.95; 3000 rows: k = 33 .. 100 0.56 .. 0.9, but 200 and 256 up to 1.1; 1500 rows up to 1.3, 1000 rows
    up to 1.5, 250 rows 3 .. 6)."""
    if not (a.dtype == torch.float32 and 32 < k <= 400 and m * n >= 2.1e6 and not 64 < n < 72 and not (k > 128 and 128 < n <= 160) and
            not (k > 256 and n <= 48)):
        return None
    turn = 1024 if k <= 192 else 2048
    if m < 2000 or (m < 4000 and 5 * m < 4 * turn * -(-m // turn)):
        return None
    return _product_operands(a, b, transposed, m, k, n)


def row_product(a, b, transposed=False, bias=None):
    """``a b`` (``transposed``: ``a b^T``) ``+ bias`` for the rows ``a`` [m, k] of a block and a layer's weight ``b`` [k, n]
    (transposed: [n, k]); fp32 sums, result in the operands' dtype."""
    if a.dim() != 2 or b.dim() != 2 or a.size(1) != b.size(1 if transposed else 0):
        raise RuntimeError("row_product: shapes %s and %s do not match" % (tuple(a.shape), tuple(b.shape)))
    m, k, n = int(a.size(0)), int(a.size(1)), int(b.size(0 if transposed else 1))
    at = _forms_row_product(a, b, transposed, m, k, n) or _forms_split_product(a, b, transposed, m, k, n)
    if at is None or not (bias is None or (bias.device == a.device and bias.dtype == a.dtype and bias.is_contiguous() and bias.numel() == n and
                                           not (torch.is_grad_enabled() and bias.requires_grad))):
        w = b.transpose(0, 1) if transposed else b
        return torch.mm(a, w) if bias is None else torch.addmm(bias, a, w)
    dev = a.device
    with _on_device(dev):
        out = torch.empty((m, n), dtype=a.dtype, device=dev)
        L.check(L.lib().fgl_row_product(*at, int(transposed), m, k, n, L.F32 if a.dtype == torch.float32 else L.BF16, L.ptr(bias), out.data_ptr(), n,
                                        L.stream_handle()))
    return out


def row_product_sum(a0, b0, a1, b1, bias=None):
    """``a0 b0^T + (a1 b1^T + bias)`` in one pass over the result, for the operands that ``row_product`` takes to the kernel; ``None`` for all
    others.  bf16: rounded where the two products and their sum would be; fp32: one sum over both products' terms, the bias added last."""
    m, n = int(a0.size(0)), int(b0.size(0))
    k0, k1 = int(a0.size(1)), int(a1.size(1))
    if int(a1.size(0)) != m or int(b1.size(0)) != n or a1.dtype != a0.dtype or a1.device != a0.device or int(b0.size(1)) != k0 or int(b1.size(1)) != k1:
        return None
    at0, at1 = _forms_row_product(a0, b0, True, m, k0, n), _forms_row_product(a1, b1, True, m, k1, n)
    if at0 is None or at1 is None or not (bias is None or (bias.device == a0.device and bias.dtype == a0.dtype and bias.is_contiguous() and
                                                           bias.numel() == n and not (torch.is_grad_enabled() and bias.requires_grad))):
        return None
    dev = a0.device
    with _on_device(dev):
        out = torch.empty((m, n), dtype=a0.dtype, device=dev)
        L.check(L.lib().fgl_row_product_sum(*at0, k0, *at1, k1, 1, m, n, L.F32 if a0.dtype == torch.float32 else L.BF16, L.ptr(bias),
                                            out.data_ptr(), n, L.stream_handle()))
    return out


def row_product_add_(out, a, b):
    """``out[:len(a)] += a b``, the product rounded before it is added; ``out`` is contiguous and nobody else's."""
    m, k, n = int(a.size(0)), int(a.size(1)), int(b.size(1))
    fits = out.dim() == 2 and out.size(0) >= m and out.size(1) == n and int(b.size(0)) == k
    at = _forms_row_product(a, b, False, m, k, n) if fits and out.dtype == a.dtype and out.device == a.device and out.is_contiguous() else None
    if at is None:
        out[:m].add_(row_product(a, b))
        return out
    with _on_device(a.device):
        L.check(L.lib().fgl_row_product_add(*at, 0, m, k, n, L.F32 if a.dtype == torch.float32 else L.BF16, out.data_ptr(), n, L.stream_handle()))
    return out


def weight_grad(a, b, column_sums=False):
    """``a^T b`` for ``a`` [k, m] and ``b`` [k, n]: a dense layer's weight gradient from its input rows and the gradient of
    its output (fp32 sums, result in the operands' dtype).  ``column_sums=True``: ``(a^T b, a.sum(0))``, with ``a`` the
    gradient of the output the transposed weight gradient and the bias gradient of the layer."""
    (k, m), n = a.shape, int(b.size(1))
    (lda, unit_a), (ldb, unit_b), at = a.stride(), b.stride(), _addresses(a, b)
    if not (a.is_cuda and a.get_device() == b.get_device() and a.dtype == b.dtype and a.dtype in _FEAT and k > 0 and m > 0 and n > 0 and
            not (torch.is_grad_enabled() and (a.requires_grad or b.requires_grad)) and  # (a graph is being built: torch's product has a gradient)
            not torch.is_autocast_enabled() and not _followed() and at is not None and
            unit_a == 1 and unit_b == 1 and m <= lda < 1 << 24 and n <= ldb < 1 << 24 and
            m < 1 << 16 and n < 1 << 16 and b.size(0) == k and
            _splits_k(k, m, n)):
        d_w = torch.mm(a.transpose(0, 1), b)
        return (d_w, a.sum(0)) if column_sums else d_w
    lib = L.lib()
    dev = a.device
    dtype = L.F32 if a.dtype == torch.float32 else L.BF16
    with _on_device(dev):
        d_w = torch.empty((m, n), dtype=a.dtype, device=dev)
        sums = torch.empty(m, dtype=a.dtype, device=dev) if column_sums else None
        ws = L.workspace(lib.fgl_weight_grad_workspace_bytes_for(k, m, n, dtype), dev)
        L.check(lib.fgl_weight_grad(at[0], lda, at[1], ldb, k, m, n, dtype, d_w.data_ptr(), n, L.ptr(sums),
                                    ws.data_ptr(), ws.numel(), L.stream_handle()))
    return (d_w, sums) if column_sums else d_w


_MODES = {"sum": L.AGG_SUM, "mean": L.AGG_MEAN, "gcn": L.AGG_GCN, "colmean": L.AGG_COLMEAN, "edge": L.AGG_EDGE,
          "colmean_ptr": L.AGG_COLMEAN_PTR, "gcn_own": L.AGG_GCN_OWN, "gcn_own_ptr": L.AGG_GCN_OWN_PTR}
_ZERO = {"self": L.ZERO_COPY_SELF, "zeros": L.ZERO_ZEROS}


def aggregate(indptr, indices, feat, mode="sum", zero_policy="self", row_norm=None, col_norm=None, n_rows=None,
              out=None, edge_weight=None, n_heads=1, edge_index=None, longest_row=None, n_rows_dev=None, mapping="auto"):
    """``out[r] = sum_e w(r, indices[e]) * feat[indices[e]]`` over the CSR rows (fp32
    accumulation; fp32 or bf16 storage).  ``mode``: sum | mean | gcn | colmean | edge | colmean_ptr (colmean with
    ``col_norm`` holding the offsets array whose differences are the counts: a block's ``edge_ptr``) | gcn_own,
    gcn_own_ptr (gcn with the rows' own entry counts as ``row_norm``, and ``col_norm`` as counts or as offsets);
    ``zero_policy``: what a row without entries gets -- ``self`` (``feat[r]``) or ``zeros``.
    ``longest_row``: what is known about the longest row's entry count -- an ``int`` bound (the fanout of a
    sampled block) or a one-element int32 device tensor (as ``block_transpose`` makes).  Speed only: hub rows
    of hundreds of entries get a second launch that a bound can save.  When not given it is taken from the
    ``fgl_longest_row`` attribute that ``block_transpose`` and the sampler attach to their ``indptr`` tensors.
    ``mode="edge"``: ``edge_weight`` float32 [n_entries, n_heads], weight of entry e for column f is
    ``edge_weight[edge_index[e] if edge_index is not None else e, f // (D // n_heads)]``.
    ``n_rows_dev``: one-element int32 device tensor with the actual row count when the host only knows the
    bound ``n_rows`` (a block whose sizes have not been read back yet): rows past it are left unwritten.
    ``mapping``: ``"auto"`` lets the library pick how lanes are dealt to rows from the row count, the entry count
    and ``longest_row`` (several lane groups per row for few long rows, several rows per group for many short
    ones); ``"row"`` asks for one lane group per row whatever the shape (what measurements of that kernel use)."""
    _check_input(indptr, "indptr", _I32)
    _check_input(indices, "indices", _I32)
    if not isinstance(feat, torch.Tensor) or not feat.is_cuda:
        raise RuntimeError("feat must be a CUDA tensor")
    if feat.dim() != 2 or feat.stride(1) != 1 or feat.dtype not in _FEAT:
        raise RuntimeError("feat must be a 2-D fp32/bf16 tensor with unit column stride")
    if row_norm is not None:
        _check_input(row_norm, "row_norm", _I32)
    if col_norm is not None:
        _check_input(col_norm, "col_norm", _I32)
    if edge_weight is not None:
        _check_input(edge_weight, "edge_weight", (torch.float32,))
        if edge_weight.dim() != 2 or edge_weight.size(1) != int(n_heads):
            raise RuntimeError("edge_weight must be [n_entries, n_heads]")
        if edge_index is None and edge_weight.size(0) < indices.numel():
            raise RuntimeError("edge_weight has fewer rows than there are entries")
    if edge_index is not None:
        _check_input(edge_index, "edge_index", _I32)
        if edge_index.numel() < indices.numel():
            raise RuntimeError("edge_index has fewer entries than indices")
    if mode == "edge" and (edge_weight is None or feat.size(1) % int(n_heads) != 0):
        raise RuntimeError("mode 'edge' needs edge_weight and a head count that divides the row length")
    if longest_row is None:
        longest_row = getattr(indptr, "fgl_longest_row", None)
    longest_host, longest_dev = -1, None
    if isinstance(longest_row, torch.Tensor):
        _check_input(longest_row, "longest_row", _I32)
        if longest_row.numel() != 1:
            raise RuntimeError("longest_row must hold one int32")
        longest_dev = longest_row
    elif longest_row is not None:
        longest_host = int(longest_row)
    if n_rows_dev is not None:
        _check_input(n_rows_dev, "n_rows_dev", _I32)
        if n_rows_dev.numel() != 1:
            raise RuntimeError("n_rows_dev must hold one int32")
    dev = _same_device(indptr, indices, feat, row_norm, col_norm, edge_weight, edge_index, longest_dev, n_rows_dev)
    n = int(indptr.numel()) - 1 if n_rows is None else int(n_rows)
    if n < 0 or n > indptr.numel() - 1:
        raise RuntimeError("n_rows (%d) does not match indptr (%d entries)" % (n, indptr.numel()))
    if mapping not in ("auto", "row"):
        raise RuntimeError("mapping must be 'auto' or 'row'")
    m = _MODES[mode]
    z = _ZERO[zero_policy]
    if z == L.ZERO_COPY_SELF and n > feat.size(0):
        raise RuntimeError("zero_policy 'self' needs feat to have a row for every output row")
    D = int(feat.size(1))
    with _on_device(dev):
        if out is None:
            out = torch.empty((n, D), dtype=feat.dtype, device=dev)
        elif out.shape != (n, D) or out.dtype != feat.dtype or out.stride(1) != 1 or not out.is_cuda:
            raise RuntimeError("out has the wrong shape, dtype or layout")
        if n > 0:
            # a block without entries has no index array to point at; the kernel then reads none
            idx_ptr = L.ptr(indices) if indices.numel() else L.ptr(indptr)
            n_entries = int(indices.numel()) if mapping == "auto" else -1
            longest_known = longest_host if mapping == "auto" else -1
            dtype = L.F32 if feat.dtype == torch.float32 else L.BF16
            ws, ws_bytes = None, 0
            if n_entries >= L.AGG_SEG_MIN_ENTRIES:
                ws_bytes = L.lib().fgl_aggregate_workspace_bytes_for(n_entries, n, int(feat.size(0)), D, dtype, m, longest_known)
                ws = L.workspace(ws_bytes, dev) if ws_bytes else None
            L.check(L.lib().fgl_aggregate_ws(L.ptr(indptr), idx_ptr, n, L.ptr(n_rows_dev), L.ptr(feat), int(feat.stride(0)), D,
                                             dtype, m, z, L.ptr(row_norm),
                                             L.ptr(col_norm), L.ptr(edge_weight), int(n_heads), L.ptr(edge_index),
                                             longest_known, L.ptr(longest_dev), n_entries, L.ptr(out),
                                             int(out.stride(0)), L.ptr(ws), ws_bytes, L.stream_handle()))
    return out


def zero_empty_rows_(indptr, x, n_rows):
    """Rows of ``x`` [n_rows, D] that have no entries in the CSR become zeros, in place."""
    with _on_device(x.device):
        L.check(L.lib().fgl_zero_empty_rows(L.ptr(indptr), int(n_rows), None, L.ptr(x), int(x.stride(0)), int(x.size(1)),
                                            L.F32 if x.dtype == torch.float32 else L.BF16, L.stream_handle()))
    return x


def head_scores(feat, attn_l, attn_r, n_dst):
    """``(el, er)`` of a GAT layer: ``el[i, h] = sum_f feat[i, h * F + f] * attn_l[h, f]`` for all rows and ``er`` with
    ``attn_r`` for the first ``n_dst`` rows, in one pass over ``feat`` (float32 [n, H * F]; attn_*: float32 [.., H, F]).
    No gradients."""
    _check_input(feat, "feat", (torch.float32,))
    _check_input(attn_l, "attn_l", (torch.float32,))
    _check_input(attn_r, "attn_r", (torch.float32,))
    H, F = int(attn_l.size(-2)), int(attn_l.size(-1))
    n, n_dst = int(feat.size(0)), int(n_dst)
    if feat.dim() != 2 or feat.size(1) != H * F or attn_l.numel() != H * F or attn_r.numel() != H * F or not 0 <= n_dst <= n:
        raise RuntimeError("feat %s does not match the attention vectors %s, %s and %d rows" % (
            tuple(feat.shape), tuple(attn_l.shape), tuple(attn_r.shape), n_dst))
    dev = _same_device(feat, attn_l, attn_r)
    with _on_device(dev):
        scores = torch.empty((n + n_dst, H), dtype=torch.float32, device=dev)
        el, er = scores[:n], scores[n:]
        if n > 0 and H * F > 0:
            L.check(L.lib().fgl_head_scores(L.ptr(feat), H * F, n, n_dst, H, F, L.ptr(attn_l), L.ptr(attn_r), L.ptr(el), L.ptr(er), L.stream_handle()))
    return el, er


def edge_softmax(indptr, indices, el, er, negative_slope=0.2, n_rows=None):
    """Attention coefficients of a GAT layer over a block CSR, ``float32 [n_entries, n_heads]``:
    ``softmax`` over the entries of each row of ``leaky_relu(el[indices[e]] + er[row])`` -- the reference's
    ``u_add_v`` + ``leaky_relu`` + ``edge_softmax`` (GraphConv.py:265-272) in one launch.  ``el``: float32
    [n_cols, n_heads], ``er``: float32 [n_rows, n_heads]."""
    _check_input(indptr, "indptr", _I32)
    _check_input(indices, "indices", _I32)
    _check_input(el, "el", (torch.float32,))
    _check_input(er, "er", (torch.float32,))
    if el.dim() != 2 or er.dim() != 2 or el.size(1) != er.size(1):
        raise RuntimeError("el and er must be [n, n_heads] with the same head count")
    dev = _same_device(indptr, indices, el, er)
    n = int(indptr.numel()) - 1 if n_rows is None else int(n_rows)
    if n < 0 or n > indptr.numel() - 1 or n > er.size(0):
        raise RuntimeError("n_rows (%d) does not match indptr (%d entries) / er (%d rows)" % (n, indptr.numel(), er.size(0)))
    H = int(el.size(1))
    with _on_device(dev):
        alpha = torch.empty((int(indices.numel()), H), dtype=torch.float32, device=dev)
        if n > 0 and indices.numel() > 0:
            L.check(L.lib().fgl_edge_softmax(L.ptr(indptr), L.ptr(indices), n, None, L.ptr(el), L.ptr(er), H,
                                             float(negative_slope), L.ptr(alpha), L.stream_handle()))
    return alpha


def block_transpose(indptr, indices, n_rows, n_cols, edge_ids=False, sorted_rows=False):
    """Column-major companion ``(t_indptr[n_cols+1], t_indices[nnz])`` of a block CSR; with
    ``edge_ids=True`` also ``t_edge[nnz]``, the position in ``indices`` of every transposed entry.
    ``sorted_rows=True`` lists every column's rows in ascending order (deterministic; the default
    leaves the order within a column to scheduling and is faster)."""
    _check_input(indptr, "indptr", _I32)
    _check_input(indices, "indices", _I32)
    dev = _same_device(indptr, indices)
    n_rows, n_cols = int(n_rows), int(n_cols)
    nnz = int(indices.numel())
    lib = L.lib()
    with _on_device(dev):
        t_ptr = torch.empty(n_cols + 1, dtype=torch.int32, device=dev)
        t_idx = torch.empty(max(nnz, 1), dtype=torch.int32, device=dev)[:nnz]
        t_edge = torch.empty(max(nnz, 1), dtype=torch.int32, device=dev)[:nnz] if edge_ids else None
        longest = torch.empty(1, dtype=torch.int32, device=dev)
        ws = L.workspace(lib.fgl_block_transpose_workspace_bytes(n_cols, nnz, int(sorted_rows)), dev)
        L.check(lib.fgl_block_transpose(L.ptr(indptr), L.ptr(indices), n_rows, None, n_cols, None, nnz, L.ptr(t_ptr),
                                        L.ptr(t_idx), L.ptr(t_edge), L.ptr(longest), int(sorted_rows), L.ptr(ws), ws.numel(),
                                        L.stream_handle()))
    t_ptr.fgl_longest_row = longest  # read by aggregate()
    return (t_ptr, t_idx, t_edge) if edge_ids else (t_ptr, t_idx)


def block_transpose_batch(blocks, edge_ids=False):
    """``block_transpose`` (unordered lists) for several blocks in the launches that one takes.  ``blocks``: list of
    ``(indptr, indices, n_rows, n_cols)``; returns a list of ``(t_indptr, t_indices, t_edge or None)`` in the same order.
    Blocks too large for the batched entry point (2^20 entries, 2^23 columns: they fill the chip on their own) are
    transposed one by one."""
    lib = L.lib()
    out = [None] * len(blocks)
    small = []
    for i, (indptr, indices, n_rows, n_cols) in enumerate(blocks):
        _check_input(indptr, "indptr", _I32)
        _check_input(indices, "indices", _I32)
        if int(indices.numel()) < L.TRANSPOSE_BATCH_MAX_EDGES and int(n_cols) < L.TRANSPOSE_BATCH_MAX_COLS:
            small.append(i)
        else:
            r = block_transpose(indptr, indices, n_rows, n_cols, edge_ids=edge_ids)
            out[i] = (r[0], r[1], r[2] if edge_ids else None)
    for g in range(0, len(small), L.TRANSPOSE_BATCH_MAX):
        group = small[g:g + L.TRANSPOSE_BATCH_MAX]
        n = len(group)
        dev = _same_device(*[blocks[i][0] for i in group], *[blocks[i][1] for i in group])
        with _on_device(dev):
            res = []
            for i in group:
                indptr, indices, n_rows, n_cols = blocks[i]
                nnz = int(indices.numel())
                t_ptr = torch.empty(int(n_cols) + 1, dtype=torch.int32, device=dev)
                t_idx = torch.empty(max(nnz, 1), dtype=torch.int32, device=dev)[:nnz]
                t_edge = torch.empty(max(nnz, 1), dtype=torch.int32, device=dev)[:nnz] if edge_ids else None
                longest = torch.empty(1, dtype=torch.int32, device=dev)
                t_ptr.fgl_longest_row = longest
                res.append((t_ptr, t_idx, t_edge, longest))
            i64 = lambda vals: (C.c_int64 * n)(*[int(v) for v in vals])
            ptrs = lambda ts: (C.c_void_p * n)(*[L.ptr(t) for t in ts])
            n_rows_a, n_cols_a = i64(blocks[i][2] for i in group), i64(blocks[i][3] for i in group)
            n_edges_a = i64(blocks[i][1].numel() for i in group)
            ws = L.workspace(lib.fgl_block_transpose_batch_workspace_bytes(n, n_cols_a, n_edges_a), dev)
            L.check(lib.fgl_block_transpose_batch(n, ptrs(blocks[i][0] for i in group), ptrs(blocks[i][1] for i in group), n_rows_a,
                                                  n_cols_a, n_edges_a, ptrs(r[0] for r in res), ptrs(r[1] for r in res),
                                                  ptrs(r[2] for r in res) if edge_ids else None, ptrs(r[3] for r in res),
                                                  L.ptr(ws), ws.numel(), L.stream_handle()))
        for i, r in zip(group, res):
            out[i] = r[:3]
    return out


def table_size(num: int, scale: int) -> int:
    """The reference's TableSize (cuda_hashtable.cuh:27-30)."""
    return int(L.lib().fgl_table_size(int(num), int(scale)))


class BlocksPlan:
    """Bounds and persistent scratch for sampling mini-batches of one shape."""

    def __init__(self, n_nodes: int, n_seeds: int, hop_fanouts, device, node_capacity=None, transpose_hops=()):
        """``node_capacity`` (optional, ``n_hops + 1`` ints): the caller's own limit on the node count
        before each hop / after the last; the worst-case bounds are clipped to it.
        ``transpose_hops``: the hops (sampling order, negative = from the end) whose transposed block
        ``sample_blocks_fused`` is to build along the way."""
        lib = L.lib()
        self.n_nodes, self.n_seeds = int(n_nodes), int(n_seeds)
        self.hop_fanouts = [int(f) for f in hop_fanouts]
        self.n_hops = len(self.hop_fanouts)
        self.device = torch.device(device)
        self._fan = (C.c_int32 * self.n_hops)(*self.hop_fanouts)
        self._node_cap = None if node_capacity is None else (C.c_int64 * (self.n_hops + 1))(*[int(c) for c in node_capacity])
        cap_dst = (C.c_int64 * self.n_hops)()
        cap_edges = (C.c_int64 * self.n_hops)()
        cap_uniq, slots, ws_bytes = C.c_int64(), C.c_int64(), C.c_size_t()
        self.transpose_hops = sorted({(int(h) + self.n_hops) % self.n_hops for h in transpose_hops})
        self.transpose_mask = sum(1 << h for h in self.transpose_hops)
        L.check(lib.fgl_sample_blocks_plan(self.n_nodes, self.n_seeds, self._fan, self.n_hops, self._node_cap, self.transpose_mask,
                                           cap_dst, cap_edges, C.byref(cap_uniq), C.byref(slots), C.byref(ws_bytes)))
        self.cap_dst = list(cap_dst)
        self.cap_edges = list(cap_edges)
        self.cap_uniq, self.slots, self.ws_bytes = cap_uniq.value, slots.value, ws_bytes.value
        self.cap_src = self.cap_dst[1:] + [self.cap_uniq]  # source nodes (columns) of each hop's block
        self.host = L.host().Plan(self.hop_fanouts, None if node_capacity is None else [int(c) for c in node_capacity], self.cap_dst,
                                  self.cap_edges, self.cap_src, self.cap_uniq, self.transpose_mask)
        self.table = torch.empty(self.slots, dtype=torch.int64, device=self.device)
        self.ws = torch.empty(max(self.ws_bytes, 256), dtype=torch.uint8, device=self.device)
        # the slot count that the last call on this plan's table left empty (None: unknown contents)
        self.empty_slots = None


_ID_ORDER = {"first": L.IDMAP_ORDERED, "arrival": L.IDMAP_ARRIVAL}


def sample_blocks_fused(plan: BlocksPlan, edge_ptr, indices, seeds, rng_seed: int, stream_base: int,
                        keep_global=(0,), table_slots=None, id_order="first", stream_offset=None, readback=None,
                        launch_stream=None, sort_transposed=False):
    """All hops of one mini-batch in one enqueue (no host synchronisation inside).

    Returns device tensors sized by the plan's bounds: ``(uniq, block_ptr[h], src_local[h],
    src_global[h] or None, counts, transposed[h])``; hop 0 expands the raw seeds.  ``counts`` (int32,
    ``3*n_hops + 2``) holds the node count before each hop and after the last, then the
    edge count of each hop, then the status word, then per hop the longest row of its transposed block
    (zero where none was built); the caller reads it once per batch.
    For the hops in ``plan.transpose_hops`` the call also builds the transposed block:
    ``transposed[h] = (t_ptr, t_dst, t_edge)`` (bound-sized; ``None`` for the other hops).
    ``keep_global`` lists the hops (negative = from the end) whose pre-relabel source ids are kept.
    ``table_slots`` (a power of two, default the plan's worst case) uses only that much of the
    hash table; a batch that outgrows it is reported in the status word (FGL_STATUS_TABLE_FULL).
    ``id_order``: ``"first"`` numbers new ids by first occurrence (deterministic), ``"arrival"`` as
    their inserts land (the reference's rule: a tenth slower where hops are small, a few per cent to an eighth faster
    from some 20 K seeds or a million edges a hop on; any run is a valid map, equal to every other after
    sorting the new ids).
    ``stream_offset``: one-element int32 device tensor added to ``stream_base`` when the kernels run (for
    callers that capture this call in a graph and advance the random stream between replays).
    ``readback``: a pinned int32 host tensor of ``3*n_hops + 2`` elements; the kernels store a copy of
    ``counts`` there when the last of them is final, so the caller's read-back is a wait for the stream and a
    look at that tensor, with no copy to enqueue.
    ``sort_transposed``: the rows of the transposed blocks come out in ascending order of their entries' positions in
    the block (run-to-run identical arrays and, with them, fp32 sums of the backward gathers; one more launch).
    ``launch_stream``: a ``torch.cuda.Stream`` to enqueue the kernels on instead of the current one (the outputs are
    still allocated on the current stream, where their consumer runs; the caller orders the two streams)."""
    _check_input(edge_ptr, "edge_ptr", _PTR)
    _check_input(indices, "indices", _I32)
    _check_input(seeds, "seeds", _I32)
    if stream_offset is not None:
        _check_input(stream_offset, "stream_offset", _I32)
    dev = _same_device(edge_ptr, indices, seeds, stream_offset)
    if int(seeds.numel()) != plan.n_seeds:
        raise RuntimeError("plan was made for %d seeds, got %d" % (plan.n_seeds, seeds.numel()))
    H = plan.n_hops
    if readback is not None and not (readback.dtype == torch.int32 and readback.is_pinned() and readback.is_contiguous()
                                     and readback.numel() >= 3 * H + 2):
        raise RuntimeError("readback must be a contiguous pinned int32 host tensor of at least %d elements" % (3 * H + 2))
    keep_mask = 0
    for h in keep_global:
        keep_mask |= 1 << ((h + H) % H)
    slots = plan.slots if table_slots is None else min(int(table_slots), plan.slots)
    # every call leaves the table empty for the next one, so only a
    # plan's first call -- or the first after a failed one, or with another slot count -- pays for a fill
    flags = _ID_ORDER[id_order] | L.BLOCKS_LEAVE_TABLE_EMPTY
    if plan.empty_slots == slots:
        flags |= L.BLOCKS_TABLE_EMPTY
    if sort_transposed:
        flags |= L.BLOCKS_SORT_TRANSPOSED
    plan.empty_slots = None
    with _on_device(dev):
        out = L.host().sample_blocks(plan.host, edge_ptr, indices, seeds, int(rng_seed) & 0xFFFFFFFFFFFFFFFF, int(stream_base) & 0xFFFFFFFF,
                                     stream_offset, keep_mask, flags, plan.table, slots, plan.ws, readback,
                                     None if launch_stream is None else launch_stream.cuda_stream)
    plan.empty_slots = slots
    return out


def rmat_keys(first_edge: int, n_edges: int, scale: int, n_nodes: int, seed: int, device) -> torch.Tensor:
    """2*n_edges symmetrised int64 keys ``row<<32 | col`` of seeded R-MAT draws (INT64_MAX = dropped)."""
    with torch.cuda.device(device):
        keys = torch.empty(2 * int(n_edges), dtype=torch.int64, device=device)
        L.check(L.lib().fgl_rmat_keys(int(first_edge), int(n_edges), int(scale), int(n_nodes),
                                      int(seed) & 0xFFFFFFFFFFFFFFFF, L.ptr(keys), L.stream_handle()))
    return keys

