"""GNN layers over the memory-aware aggregation operators, with the class names, call
signatures and autograd wiring of the reference's GraphConv.py (MA_Function, GCNConv, GCN,
MA_Function_GIN, GINConv, GIN, MA_Function_GAT, GATConv, GAT; GraphConv.py:19-312), plus a mean
aggregator (GraphSAGE), which the reference's benchmark configurations name but its kernels do
not provide.

The reference's quirks are kept where they define results: weights are drawn from
U(-1/sqrt(out), 1/sqrt(out)) (GraphConv.py:52-55), dropout sits between layers, no activation
is applied by GCN / GIN (the ``activation`` argument is ignored, GraphConv.py:69,86-99), the
backward of GCN receives (dst_norm, src_norm) in the slots the extension calls
(src_norm_degs, dst_norm_degs) (GraphConv.py:37), and destination rows without edges pass
their input through in the forward pass and receive no gradient from it.
"""
from __future__ import annotations

import math

import torch
from torch import nn

from . import ops
from .sampler import Block


def _transposed(t, edge_ids=False):
    """The transposed block behind the ``transposed`` argument of the autograd functions: either the tuple
    itself or a ``Block``, whose transpose is built here, on first use in a backward pass."""
    if isinstance(t, Block):
        return t.transposed(edge_ids=True) if edge_ids else t.transposed()
    return t


def _block_csr(graph):
    """(edge_ptr, src_edges, raw_dst_degs) of a block.  A ``Block`` carries its CSR; any other
    object with ``edges()`` goes through cal_deg + exclusive_sum like GraphConv.py:93-98."""
    dst_nodes = graph.num_dst_nodes()
    if isinstance(graph, Block):
        return graph.edge_ptr, graph.src_local, graph.in_degrees()
    raw = ops.cal_deg(graph.edges()[1].int(), dst_nodes)
    return ops.exclusive_sum(raw), graph.edges()[0].int(), raw


def _aggregate_first_is_cheaper(n_src, n_dst, n_edges, d_in, d_out):
    """(A X) W against A (X W): the product runs over n_dst rows instead of n_src, the gather moves rows of
    d_in instead of d_out columns.  Priced with round figures for this GPU (fp32 matrix product ~50 TFLOP/s,
    random row gather ~5 TB/s); the two orders agree up to fp32 rounding."""
    flop_s, byte_s = 50e12, 5e12
    product_first = 2.0 * n_src * d_in * d_out / flop_s + 4.0 * n_edges * d_out / byte_s
    gather_first = 2.0 * n_dst * d_in * d_out / flop_s + 4.0 * n_edges * d_in / byte_s
    return gather_first < product_first


class MA_Function(torch.autograd.Function):
    """GCN layer ``A_norm X W``.  The reference multiplies first and gathers rows of ``X W``
    (aggregate_acc.cpp:133-160); a sampled block has several times more source than destination rows, so
    for most layers it is cheaper to gather rows of ``X`` and multiply the (fewer) gathered rows --
    ``order="auto"`` (default) prices both and picks; ``"product_first"`` is the reference's order.  Either
    way a destination row without edges passes ``(X W)[d]`` through and sends no gradient back
    (aggregate_acc_kernel.cu:307-309,498-500).
    ``src_norm_degs`` and ``dst_norm_degs`` may be ``None`` when ``transposed`` is the ``Block`` itself: its degrees are
    then read from its row pointers, with no arrays made of them (what ``GCN`` does: six launches per layer less)."""

    @staticmethod
    def _gather(edge_ptr, src_edges, feat, src_norm_degs, dst_norm_degs, n_dst, block, zero_policy, longest_row):
        if src_norm_degs is not None:
            mode, row_norm, col_norm = "gcn", dst_norm_degs, src_norm_degs
        elif block._transposed is not None:
            mode, row_norm, col_norm = "gcn_own_ptr", None, block._transposed[0]
        else:
            mode, row_norm, col_norm = "gcn_own", None, block.out_degrees()
        return ops.aggregate(edge_ptr, src_edges, feat, mode=mode, zero_policy=zero_policy, row_norm=row_norm, col_norm=col_norm,
                             n_rows=n_dst, longest_row=longest_row)

    @staticmethod
    def _gather_back(t_ptr, t_idx, d_out, src_norm_degs, dst_norm_degs, n_src, edge_ptr):
        if src_norm_degs is not None:
            return ops.aggregate(t_ptr, t_idx, d_out, mode="gcn", zero_policy="zeros", row_norm=src_norm_degs, col_norm=dst_norm_degs, n_rows=n_src)
        return ops.aggregate(t_ptr, t_idx, d_out, mode="gcn_own_ptr", zero_policy="zeros", col_norm=edge_ptr, n_rows=n_src)

    @staticmethod
    def forward(ctx, edge_ptr, src_edges, src_norm_degs, dst_norm_degs, dst_nodes, input_feat, weight, neighbor_num,
                transposed=None, order="auto"):
        ctx.transposed = transposed
        n_dst = int(dst_nodes)
        gather_first = order == "gather_first" or (order == "auto" and _aggregate_first_is_cheaper(
            input_feat.size(0), n_dst, src_edges.numel(), weight.size(0), weight.size(1)))
        ctx.gather_first = gather_first
        longest = ops._fanout_bound(edge_ptr, neighbor_num)
        if not gather_first:
            ctx.save_for_backward(edge_ptr, src_edges, src_norm_degs, dst_norm_degs, weight, input_feat)
            return MA_Function._gather(edge_ptr, src_edges, ops.row_product(input_feat, weight), src_norm_degs, dst_norm_degs, n_dst, transposed,
                                       "self", longest)
        ax = MA_Function._gather(edge_ptr, src_edges, input_feat, src_norm_degs, dst_norm_degs, n_dst, transposed, "self", longest)
        ctx.n_src = int(input_feat.size(0))
        ctx.save_for_backward(edge_ptr, src_edges, src_norm_degs, dst_norm_degs, weight, ax)
        return ops.row_product(ax, weight)

    @staticmethod
    def backward(ctx, d_input):
        d_input = d_input.contiguous()
        if ctx.gather_first:
            edge_ptr, src_edges, src_norm_degs, dst_norm_degs, weight, ax = ctx.saved_tensors
            # what the weight gradient wants of the gathered rows (nobody else has them): rows without edges send no gradient
            # back.  Here and not in forward, where a pass that records nothing would pay for it (two launches of infer's twenty).
            ops.zero_empty_rows_(edge_ptr, ax, int(d_input.size(0)))
            d_w = ops.weight_grad(ax, d_input)
            d_x = None
            if ctx.needs_input_grad[5]:
                d_ax = ops.row_product(d_input, weight, transposed=True)  # (rows without edges are in no source's list)
                if ctx.transposed is None:
                    t_ptr, t_idx = ops.block_transpose(edge_ptr, src_edges, int(d_input.size(0)), ctx.n_src)
                else:
                    t_ptr, t_idx = _transposed(ctx.transposed)
                d_x = MA_Function._gather_back(t_ptr, t_idx, d_ax, src_norm_degs, dst_norm_degs, ctx.n_src, edge_ptr)
            return None, None, None, None, None, d_x, d_w, None, None, None
        edge_ptr, src_edges, src_norm_degs, dst_norm_degs, weight, input_feat = ctx.saved_tensors
        if ctx.transposed is None:
            d_x, d_w = ops.backward_gcn(edge_ptr, src_edges, dst_norm_degs, src_norm_degs, d_input, weight, input_feat)
        elif not ctx.needs_input_grad[5]:
            # the first layer: nobody wants d_x, and d_w = X^T (A^T d_out) = (A X)^T d_out needs no transposed
            # block -- one more forward-direction gather (rows without edges contribute nothing, as in the
            # reference's backward kernel, aggregate_acc_kernel.cu:498-500)
            ax = MA_Function._gather(edge_ptr, src_edges, input_feat, src_norm_degs, dst_norm_degs, int(d_input.size(0)), ctx.transposed,
                                     "zeros", None)
            d_x, d_w = None, ops.weight_grad(ax, d_input)
        else:  # same arithmetic as backward_gcn, with the block's cached transpose
            t_ptr, t_idx = _transposed(ctx.transposed)
            g = MA_Function._gather_back(t_ptr, t_idx, d_input, src_norm_degs, dst_norm_degs, int(input_feat.size(0)), edge_ptr)
            d_x = ops.row_product(g, weight, transposed=True)
            d_w = ops.weight_grad(input_feat, g)
        return None, None, None, None, None, d_x, d_w, None, None, None


class _Conv(nn.Module):
    def __init__(self, input_dim, output_dim, weight=False):
        super().__init__()
        if weight:
            self.weights = nn.Parameter(torch.randn(input_dim, output_dim))
        else:
            self.weights = self.register_parameter('weight', None)
        self.reset_parameters()

    def reset_parameters(self):
        if self.weights is not None:
            stdv = 1. / math.sqrt(self.weights.size(1))
            self.weights.data.uniform_(-stdv, stdv)

    def _weight(self):
        if self.weights is None:
            raise RuntimeError("layer was built with weight=False")
        return self.weights


class GCNConv(_Conv):
    order = "auto"  # "product_first": the reference's order of product and gather in every layer (see MA_Function)

    def forward(self, edge_ptr, src_edges, src_norm_degs, dst_norm_degs, dst_nodes, input_feat, neighbor_num,
                transposed=None):
        return MA_Function.apply(edge_ptr, src_edges, src_norm_degs, dst_norm_degs, dst_nodes, input_feat,
                                 self._weight(), neighbor_num, transposed, self.order)


def _stack(conv, in_feats, n_hidden, n_classes, n_layers, weight):
    layers = nn.ModuleList()
    layers.append(conv(in_feats, n_hidden, weight=weight))
    for _ in range(1, n_layers - 1):
        layers.append(conv(n_hidden, n_hidden, weight=weight))
    layers.append(conv(n_hidden, n_classes, weight=weight))
    return layers


class GCN(nn.Module):
    def __init__(self, in_feats, n_hidden, n_classes, n_layers, activation, weight, dropout):
        super().__init__()
        self.layers = _stack(GCNConv, in_feats, n_hidden, n_classes, n_layers, weight)
        self.dropout = nn.Dropout(p=dropout)

    def forward(self, blocks, features, neighbor_list=[5, 10, 15]):
        h = features
        for i, layer in enumerate(self.layers):
            if i != 0:
                h = self.dropout(h)
            graph = blocks[i]
            dst_nodes = graph.num_dst_nodes()
            if isinstance(graph, Block):
                edge_ptr, src_edges, transposed = graph.edge_ptr, graph.src_local, graph  # (degrees from its row pointers)
                src_norm_degs = dst_norm_degs = None
            else:
                edge_ptr, src_edges, raw_dst_norm_degs = _block_csr(graph)
                src_norm_degs = ops.cal_deg(src_edges, graph.num_src_nodes()).clamp(min=1)
                dst_norm_degs = raw_dst_norm_degs.clamp(min=1)
                transposed = None
            h = layer(edge_ptr, src_edges, src_norm_degs, dst_norm_degs, dst_nodes, h, neighbor_list[i], transposed)
        return h


class MA_Function_GIN(torch.autograd.Function):
    @staticmethod
    def forward(ctx, edge_ptr, src_edges, dst_nodes, input_feat, weight, neighbor_num, transposed=None):
        X_prime, tmp = ops.forwaed_gin(edge_ptr, src_edges, input_feat, weight, neighbor_num, dst_nodes)
        ctx.src_nodes = input_feat.size(0)
        ctx.neighbor_num = neighbor_num
        ctx.transposed = transposed
        ctx.save_for_backward(edge_ptr, src_edges, weight, tmp)
        return X_prime

    @staticmethod
    def backward(ctx, d_input):
        edge_ptr, src_edges, weight, tmp = ctx.saved_tensors
        d_input = d_input.contiguous()
        if ctx.transposed is None:
            d_x, d_w = ops.backward_gin(edge_ptr, src_edges, d_input, weight, tmp, ctx.src_nodes)
        else:
            d_w = ops.weight_grad(tmp, d_input)
            d_x = None
            if ctx.needs_input_grad[3]:  # not for the first layer: its transposed block is never built
                t_ptr, t_idx = _transposed(ctx.transposed)
                d_tmp = ops.row_product(d_input, weight, transposed=True)
                d_x = ops.aggregate(t_ptr, t_idx, d_tmp, mode="sum", zero_policy="zeros", n_rows=int(ctx.src_nodes))
        return None, None, None, d_x, d_w, None, None


class GINConv(_Conv):
    def forward(self, edge_ptr, src_edges, dst_nodes, input_feat, neighbor_num, transposed=None):
        return MA_Function_GIN.apply(edge_ptr, src_edges, dst_nodes, input_feat, self._weight(), neighbor_num, transposed)


class GIN(nn.Module):
    def __init__(self, in_feats, n_hidden, n_classes, n_layers, activation, weight, dropout):
        super().__init__()
        self.layers = _stack(GINConv, in_feats, n_hidden, n_classes, n_layers, weight)
        self.dropout = nn.Dropout(p=dropout)

    def forward(self, blocks, features, neighbor_list=[5, 10, 15]):
        h = features
        for i, layer in enumerate(self.layers):
            if i != 0:
                h = self.dropout(h)
            graph = blocks[i]
            dst_nodes = graph.num_dst_nodes()
            edge_ptr, src_edges = (graph.edge_ptr, graph.src_local) if isinstance(graph, Block) else _block_csr(graph)[:2]
            transposed = graph if isinstance(graph, Block) and torch.is_grad_enabled() else None
            h = layer(edge_ptr, src_edges, dst_nodes, h, neighbor_list[i], transposed)
        return h


# ---------------------------------------------------------------------------------------
# dense layers
# ---------------------------------------------------------------------------------------
class _LinearFunction(torch.autograd.Function):
    """``x W^T + b`` whose weight and bias gradients come from one pass over the output's gradient (ops.weight_grad)."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        ctx.save_for_backward(x, weight)
        ctx.with_bias = bias is not None
        return ops.row_product(x, weight, transposed=True, bias=bias)

    @staticmethod
    def backward(ctx, d_out):
        x, weight = ctx.saved_tensors
        d_x = d_w = d_b = None
        if ctx.needs_input_grad[0]:
            d_x = ops.row_product(d_out, weight)
        want_bias = ctx.with_bias and ctx.needs_input_grad[2]
        if torch.is_grad_enabled():  # (a graph of the gradients is being built: operators that have gradients themselves)
            d_w = torch.mm(d_out.transpose(0, 1), x)
            d_b = d_out.sum(0) if want_bias else None
        elif ctx.needs_input_grad[1] and want_bias:
            d_w, d_b = ops.weight_grad(d_out, x, column_sums=True)
        elif ctx.needs_input_grad[1]:
            d_w = ops.weight_grad(d_out, x)
        elif want_bias:
            d_b = d_out.sum(0)
        return d_x, d_w, d_b


def _watched(t):
    """Whether the operators that ``t`` goes through are its class's business (for what else may follow them see ``ops._followed``)."""
    return type(t) not in (torch.Tensor, nn.Parameter)


class _Linear(nn.Linear):
    """``nn.Linear`` with ``_LinearFunction``'s backward pass for the inputs it is made for: plain matrices on the GPU in the
    weight's own type (fp32 or bf16), outside autocast, tracing, compilation, modes that follow the operators and forward-mode
    differentiation (``_LinearFunction`` has no rule for those; the operator has)."""

    def forward(self, x):
        # (compilation and tracing first: the compiler cannot look into the other questions)
        if torch.compiler.is_compiling() or torch.jit.is_tracing() or \
                not (x.is_cuda and x.dim() == 2 and x.dtype == self.weight.dtype and x.dtype in ops._FEAT and not torch.is_autocast_enabled()) or \
                _watched(x) or _watched(self.weight) or (self.bias is not None and _watched(self.bias)) or \
                torch.autograd.forward_ad._current_level >= 0 or ops._followed():
            return super().forward(x)
        if not torch.is_grad_enabled():
            return ops.row_product(x, self.weight, transposed=True, bias=self.bias)
        return _LinearFunction.apply(x, self.weight, self.bias)


# ---------------------------------------------------------------------------------------
# attention-weighted aggregation (GAT; GraphConv.py:198-312)
# ---------------------------------------------------------------------------------------
class MA_Function_GAT(torch.autograd.Function):
    @staticmethod
    def forward(ctx, edge_ptr, edge_data, src_edges, dst_edges, dst_nodes, input_feat, num_heads, neighbor_num,
                transposed=None):
        X_prime = ops.forward_gat(edge_ptr, edge_data, src_edges, input_feat, neighbor_num, dst_nodes, num_heads)[0]
        ctx.src_nodes = input_feat.size(0)
        ctx.num_heads = num_heads
        ctx.neighbor_num = neighbor_num
        ctx.transposed = transposed
        ctx.save_for_backward(edge_ptr, edge_data, src_edges, dst_edges, input_feat)
        return X_prime

    @staticmethod
    def backward(ctx, d_input):
        edge_ptr, edge_data, src_edges, dst_edges, input_feat = ctx.saved_tensors
        d_input = d_input.contiguous()
        if ctx.transposed is None:
            d_x = ops.backward_gat(edge_ptr, edge_data, src_edges, d_input, ctx.src_nodes, ctx.num_heads)[0]
        elif not ctx.needs_input_grad[5]:
            d_x = None
        else:
            t_ptr, t_idx, t_edge = _transposed(ctx.transposed, edge_ids=True)
            d_x = ops.aggregate(t_ptr, t_idx, d_input, mode="edge", zero_policy="zeros", n_rows=int(ctx.src_nodes),
                                edge_weight=edge_data, n_heads=int(ctx.num_heads), edge_index=t_edge)
        # as in the reference (GraphConv.py:227) the attention weights receive no gradient from here
        return None, None, None, None, None, d_x, None, None, None


def edge_softmax_torch(edge_ptr, dst_edges, e, n_dst):
    """softmax of the edge scores ``e`` [E, H] over the edges of each destination (what the reference
    takes from dgl.nn.functional.edge_softmax, GraphConv.py:272), written with torch operators: the plain
    fp32 restatement that ``ops.edge_softmax`` (one HIP launch, used by ``GATConv``) is tested against."""
    idx = dst_edges.long()
    top = torch.full((n_dst, e.size(1)), float("-inf"), dtype=e.dtype, device=e.device)
    top = top.scatter_reduce(0, idx[:, None].expand(-1, e.size(1)), e, reduce="amax", include_self=True)
    ex = torch.exp(e - top.index_select(0, idx))
    den = torch.zeros_like(top).index_add_(0, idx, ex)
    return ex / den.index_select(0, idx)


class GATConv(nn.Module):
    def __init__(self, input_dim, output_dim, num_heads, feat_drop=0, attn_drop=0, negative_slope=0.2):
        super().__init__()
        self.out_feats = output_dim
        self.num_heads = num_heads
        self.fc = _Linear(input_dim, output_dim * num_heads, bias=False)
        self.attn_l = nn.Parameter(torch.empty(1, num_heads, output_dim))
        self.attn_r = nn.Parameter(torch.empty(1, num_heads, output_dim))
        self.feat_drop = nn.Dropout(feat_drop)
        self.attn_drop = nn.Dropout(attn_drop)
        self.leaky_relu = nn.LeakyReLU(negative_slope)
        self.reset_parameters()

    def reset_parameters(self):
        gain = nn.init.calculate_gain('relu')
        nn.init.xavier_normal_(self.fc.weight, gain=gain)
        nn.init.xavier_normal_(self.attn_l, gain=gain)
        nn.init.xavier_normal_(self.attn_r, gain=gain)

    def _scores(self, feat_src, dst_nodes):
        """el [n_src, H] and er [n_dst, H].  One pass over the fp32 rows; other types (autocast, a bf16 layer) take the two
        products and sums that it replaces (105 K rows of 4 x 64 columns: 200 us)."""
        if (feat_src.is_cuda and feat_src.dtype == torch.float32 and self.attn_l.dtype == torch.float32 and self.attn_r.dtype == torch.float32
                and feat_src.is_contiguous() and self.attn_l.is_contiguous() and self.attn_r.is_contiguous() and self.attn_l.size(0) == 1
                and self.attn_r.size(0) == 1 and not ops._followed()):
            return ops.head_scores(feat_src, self.attn_l, self.attn_r, dst_nodes)
        feat_src = feat_src.view(-1, self.num_heads, self.out_feats)
        return (feat_src * self.attn_l).sum(dim=-1).contiguous(), (feat_src[:dst_nodes] * self.attn_r).sum(dim=-1).contiguous()

    def forward(self, graph, input_feat, neighbor_num):
        dst_nodes = graph.num_dst_nodes()
        feat_src = self.fc(input_feat).reshape(-1, self.out_feats * self.num_heads)  # (any leading shape of the input)
        edge_ptr, src_edges = (graph.edge_ptr, graph.src_local) if isinstance(graph, Block) else _block_csr(graph)[:2]
        # u_add_v + leaky_relu + edge_softmax (DGL calls in the reference, GraphConv.py:265-272) in one launch.
        # No gradient reaches the coefficients (the aggregation's backward returns none for them, as in the
        # reference, GraphConv.py:227), so they are computed outside the autograd graph.
        with torch.no_grad():
            el, er = self._scores(feat_src.detach(), dst_nodes)
            alpha = ops.edge_softmax(edge_ptr, src_edges, el, er, self.leaky_relu.negative_slope, n_rows=dst_nodes)
            edge_data = self.attn_drop(alpha).contiguous()
        transposed = graph if isinstance(graph, Block) and torch.is_grad_enabled() else None
        return MA_Function_GAT.apply(edge_ptr, edge_data, src_edges, None, dst_nodes, feat_src, self.num_heads,
                                     neighbor_num, transposed)


class GAT(nn.Module):
    def __init__(self, in_feats, n_hidden, n_classes, n_layers, activation, dropout, heads=8):
        super().__init__()
        self.layers = nn.ModuleList()
        self.layers.append(GATConv(in_feats, n_hidden, num_heads=heads))
        for _ in range(1, n_layers - 1):
            self.layers.append(GATConv(n_hidden * heads, n_hidden, num_heads=heads, feat_drop=dropout))
        self.layers.append(GATConv(n_hidden * heads, n_classes, num_heads=1, feat_drop=dropout))
        self.dropout = nn.Dropout(p=dropout)

    def forward(self, blocks, features, neighbor_list=[5, 10, 15]):
        h = features
        for i, layer in enumerate(self.layers):
            h = layer(blocks[i], h, neighbor_list[i])
        return h


# ---------------------------------------------------------------------------------------
# mean aggregation (GraphSAGE-mean)
# ---------------------------------------------------------------------------------------
class MA_Function_Mean(torch.autograd.Function):
    """``out[d] = mean of feat[src] over the edges into d`` (zeros if there are none).
    ``indices`` may hold block-local ids (``feat`` = the block's source rows) or graph ids
    (``feat`` = the whole resident feature table: the input-row gather fused into the first
    layer).  The gradient w.r.t. ``feat`` is produced only in the block-local form."""

    @staticmethod
    def forward(ctx, block, feat, use_global):
        indices = block.src_global if use_global else block.src_local
        ctx.block = block
        ctx.use_global = use_global
        ctx.n_src = block.num_src_nodes()
        return ops.aggregate(block.edge_ptr, indices, feat, mode="mean", zero_policy="zeros", n_rows=block.num_dst_nodes())

    @staticmethod
    def backward(ctx, d_out):
        if ctx.use_global or not ctx.needs_input_grad[1]:
            return None, None, None
        block = ctx.block
        t_ptr, t_idx = block.transposed()
        # (the destination rows' entry counts are the differences of the block's own row pointer: no degree array)
        d_feat = ops.aggregate(t_ptr, t_idx, d_out.contiguous(), mode="colmean_ptr", zero_policy="zeros",
                               col_norm=block.edge_ptr, n_rows=ctx.n_src)
        return None, d_feat, None


class _SageFunction(torch.autograd.Function):
    """A ``SAGEConv`` layer as a whole: the two products and their sum are one pass over the output, and in the backward pass the
    gradient of a node's own row is added to its row of the gathered gradient, where autograd would write it into a cleared array of all
    source rows and add that.  (GraphSAGE in bf16, 87 K and 41 K rows of 256 columns: 12 of a training step's 61 launches.)
    ``feat_dst`` is ``None`` where the destination rows are the first rows of ``feat_src``; otherwise ``feat_src`` gets no gradient (it is
    the whole table, or wants none)."""

    @staticmethod
    def run(block, feat_src, feat_dst, w_self, w_neigh, bias, use_global):
        n_dst = block.num_dst_nodes()
        h = ops.aggregate(block.edge_ptr, block.src_global if use_global else block.src_local, feat_src, mode="mean", zero_policy="zeros", n_rows=n_dst)
        x = feat_src[:n_dst] if feat_dst is None else feat_dst
        out = ops.row_product_sum(x, w_self, h, w_neigh, bias)
        if out is None:  # (sizes that are the library's)
            out = ops.row_product(x, w_self, transposed=True) + ops.row_product(h, w_neigh, transposed=True, bias=bias)
        return out, h

    @staticmethod
    def forward(ctx, block, feat_src, feat_dst, w_self, w_neigh, bias, use_global):
        out, h = _SageFunction.run(block, feat_src, feat_dst, w_self, w_neigh, bias, use_global)
        ctx.block, ctx.own_rows = block, feat_dst is None
        # (the input that the own rows come from, not the slice of it: what is saved of an input has its history when it comes back)
        ctx.save_for_backward(feat_src if feat_dst is None else feat_dst, h, w_self, w_neigh)
        return out

    @staticmethod
    def backward(ctx, d_out):
        own, h, w_self, w_neigh = ctx.saved_tensors
        _, need_src, need_dst, need_self, need_neigh, need_bias, _ = ctx.needs_input_grad
        need_src = need_src and ctx.own_rows
        d_src = d_dst = d_self = d_neigh = d_bias = None
        x = own[:ctx.block.num_dst_nodes()] if ctx.own_rows else own
        recorded = torch.is_grad_enabled()  # (a graph of the gradients is being built: operators that have gradients themselves)
        if recorded:
            if need_src and need_neigh:
                h = MA_Function_Mean.apply(ctx.block, own, False)  # (the saved one was formed inside this function: no history)
            d_self = torch.mm(d_out.transpose(0, 1), x) if need_self else None
            d_neigh = torch.mm(d_out.transpose(0, 1), h) if need_neigh else None
            d_bias = d_out.sum(0) if need_bias else None
        else:
            if need_neigh and need_bias:
                d_neigh, d_bias = ops.weight_grad(d_out, h, column_sums=True)
            elif need_neigh:
                d_neigh = ops.weight_grad(d_out, h)
            elif need_bias:
                d_bias = d_out.sum(0)
            if need_self:
                d_self = ops.weight_grad(d_out, x)
        if need_src:
            t_ptr, t_idx = ctx.block.transposed()
            d_src = ops.aggregate(t_ptr, t_idx, ops.row_product(d_out, w_neigh).contiguous(), mode="colmean_ptr", zero_policy="zeros",
                                  col_norm=ctx.block.edge_ptr, n_rows=ctx.block.num_src_nodes())
            if recorded:
                n_dst = int(d_out.size(0))
                d_src = torch.cat([d_src[:n_dst] + torch.mm(d_out, w_self), d_src[n_dst:]])
            else:
                ops.row_product_add_(d_src, d_out, w_self)
        if need_dst:
            d_dst = ops.row_product(d_out, w_self)
        return None, d_src, d_dst, d_self, d_neigh, d_bias, None


_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")


def _called_plainly(module):
    """Whether calling ``module`` runs its class's ``forward`` and nothing else."""
    d = module.__dict__
    return not any(d[k] for k in _HOOKS) and "forward" not in d and d.get("_compiled_call_impl") is None and not any(
        getattr(torch.nn.modules.module, "_global" + k) for k in _HOOKS)


class SAGEConv(nn.Module):
    """``h_dst W_self + mean(h_src) W_neigh + b`` (the mean aggregator of GraphSAGE)."""

    def __init__(self, input_dim, output_dim, bias=True):
        super().__init__()
        self.fc_self = _Linear(input_dim, output_dim, bias=False)
        self.fc_neigh = _Linear(input_dim, output_dim, bias=bias)

    def _as_one(self, block, feat_src, feat_dst, use_global):
        """Whether the layer may be formed as a whole: both parts are what ``__init__`` made them, called by nobody but this layer, their
        inputs the ones that ``_Linear`` takes to the kernels, and there is one own row for each destination (a single one that stands for
        all of them is repeated by the operators' sum) and, if they are taken from the source rows, a row of their gradient for each.
        Source rows that have a gradient are saved for gradients of the gradients; the parts save their products' inputs, no more, so where
        the own rows come from elsewhere, or a hook is handed what is saved, the layer is formed part by part."""
        if torch.compiler.is_compiling() or torch.jit.is_tracing():
            return False
        if torch.is_grad_enabled() and ((feat_dst is not None and not use_global and feat_src.requires_grad) or
                                        torch._C._autograd._top_saved_tensors_default_hooks(False) is not None):
            return False
        a, b = self.fc_self, self.fc_neigh
        if type(a) is not _Linear or type(b) is not _Linear or a.bias is not None or not _called_plainly(a) or not _called_plainly(b):
            return False
        own = feat_src if feat_dst is None else feat_dst
        n_dst = block.num_dst_nodes()
        if own.dim() != 2 or (n_dst > min(own.size(0), block.num_src_nodes()) if feat_dst is None else own.size(0) != n_dst):
            return False
        used = (feat_src, own, a.weight, b.weight) if b.bias is None else (feat_src, own, a.weight, b.weight, b.bias)
        return (feat_src.is_cuda and feat_src.dim() == 2 and feat_src.dtype in ops._FEAT and
                (feat_dst is not None or not use_global) and all(t.dtype == feat_src.dtype and t.device == feat_src.device for t in used) and
                not any(map(_watched, used)) and not torch.is_autocast_enabled() and torch.autograd.forward_ad._current_level < 0 and
                not ops._followed())

    def forward(self, block, feat_src, feat_dst=None, use_global=False):
        if isinstance(block, Block) and self._as_one(block, feat_src, feat_dst, use_global):
            args = (block, feat_src, feat_dst, self.fc_self.weight, self.fc_neigh.weight, self.fc_neigh.bias, use_global)
            return _SageFunction.apply(*args) if torch.is_grad_enabled() else _SageFunction.run(*args)[0]
        h_neigh = MA_Function_Mean.apply(block, feat_src, use_global)
        if feat_dst is None:
            feat_dst = feat_src[:block.num_dst_nodes()]
        return self.fc_self(feat_dst) + self.fc_neigh(h_neigh)


class SAGE(nn.Module):
    def __init__(self, in_feats, n_hidden, n_classes, n_layers, activation=torch.relu, dropout=0.0):
        super().__init__()
        dims = [in_feats] + [n_hidden] * (n_layers - 1) + [n_classes]
        self.layers = nn.ModuleList(SAGEConv(dims[i], dims[i + 1]) for i in range(n_layers))
        self.activation = activation
        self.dropout = nn.Dropout(p=dropout)

    def forward(self, blocks, features, input_nodes=None):
        """``features``: the rows of the input nodes, or -- with ``input_nodes`` given -- the
        whole feature table, in which case the first layer gathers straight from it."""
        h = features
        for i, (layer, block) in enumerate(zip(self.layers, blocks)):
            if i == 0 and input_nodes is not None:
                if block.src_global is None:
                    raise RuntimeError("the outermost block does not carry graph ids")
                dst_ids = input_nodes[:block.num_dst_nodes()]
                if dst_ids.dtype != torch.int32 or features.requires_grad:
                    dst_ids = dst_ids.long()
                h = layer(block, features, feat_dst=features.index_select(0, dst_ids), use_global=True)
            else:
                h = layer(block, h)
            if i != len(self.layers) - 1:
                if self.activation is not None:
                    h = self.activation(h)
                h = self.dropout(h)
        return h
