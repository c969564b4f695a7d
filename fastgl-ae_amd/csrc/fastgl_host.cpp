// Host half of the fused sampling call for the Python package (fastgl/ops.py, fastgl/sampler.py): the outputs of a mini-batch
// are allocated, handed to fgl_sample_blocks and cut to their sizes here.
//
// A mini-batch of three hops has 15 output arrays.  From Python their allocation, the pointer arrays and the 40 arguments of the
// call, and the 13 views at the end, cost more host time than the 8 launches they surround, and the GPU waits for them: nothing is
// enqueued before the arrays exist, and the next mini-batch starts behind the views.
//
// Host code only (g++ against the torch headers, linked with libfastgl_hip.so): torch owns the memory and names the stream.
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#include <string>
#include <vector>

#include "fastgl_hip.h"

namespace {

// bounds of the mini-batches of one shape (ops.BlocksPlan)
struct Plan {
    std::vector<int32_t> fanouts;
    std::vector<int64_t> node_capacity;  // empty: none
    std::vector<int64_t> cap_dst, cap_edges, cap_src;
    int64_t cap_uniq;
    uint32_t transpose_mask;
};

using Maybe = c10::optional<torch::Tensor>;

void* address(const Maybe& t) { return t.has_value() ? t->data_ptr() : nullptr; }

// ops.sample_blocks_fused behind its checks; launch_stream: a stream to enqueue on instead of the current one, or null
py::tuple sample_blocks(const Plan& p, const torch::Tensor& edge_ptr, const torch::Tensor& indices, const torch::Tensor& seeds,
                        uint64_t rng_seed, uint32_t stream_base, const Maybe& stream_offset, uint32_t keep_mask, int flags,
                        const torch::Tensor& table, int64_t slots, const torch::Tensor& ws, const Maybe& readback,
                        c10::optional<uint64_t> launch_stream)
{
    const size_t n_hops = p.fanouts.size();
    const auto like = seeds.options();
    auto array = [&](int64_t n) { return torch::empty({n}, like); };
    auto at_least_one = [](int64_t n) { return n > 1 ? n : (int64_t)1; };
    torch::Tensor uniq = array(at_least_one(p.cap_uniq));
    std::vector<torch::Tensor> block_ptr(n_hops), src_local(n_hops), t_ptr(n_hops), t_dst(n_hops), t_edge(n_hops);
    std::vector<Maybe> src_global(n_hops);
    std::vector<int32_t*> a[6];
    for (auto& v : a) v.assign(n_hops, nullptr);
    for (size_t h = 0; h < n_hops; ++h) {
        block_ptr[h] = array(p.cap_dst[h] + 1);
        src_local[h] = array(at_least_one(p.cap_edges[h]));
        a[0][h] = block_ptr[h].data_ptr<int32_t>();
        a[1][h] = src_local[h].data_ptr<int32_t>();
        if ((keep_mask >> h) & 1u) {
            src_global[h] = array(at_least_one(p.cap_edges[h]));
            a[2][h] = src_global[h]->data_ptr<int32_t>();
        }
        if ((p.transpose_mask >> h) & 1u) {
            t_ptr[h] = array(p.cap_src[h] + 1);
            t_dst[h] = array(at_least_one(p.cap_edges[h]));
            t_edge[h] = array(at_least_one(p.cap_edges[h]));
            a[3][h] = t_ptr[h].data_ptr<int32_t>();
            a[4][h] = t_dst[h].data_ptr<int32_t>();
            a[5][h] = t_edge[h].data_ptr<int32_t>();
        }
    }
    torch::Tensor counts = array(3 * (int64_t)n_hops + 2);
    const bool transposed = p.transpose_mask != 0;
    void* stream = launch_stream.has_value() ? reinterpret_cast<void*>(*launch_stream)
                                             : static_cast<void*>(c10::hip::getCurrentHIPStream(seeds.get_device()).stream());
    const void* indptr = edge_ptr.data_ptr();
    const int is64 = edge_ptr.scalar_type() == torch::kInt64;
    void* table_ptr = table.data_ptr();
    void* ws_ptr = ws.data_ptr();
    int rc;
    std::string error;
    {
        py::gil_scoped_release released;
        rc = fgl_sample_blocks(indptr, is64, indices.data_ptr<int32_t>(), edge_ptr.numel() - 1, seeds.data_ptr<int32_t>(), seeds.numel(),
                               p.fanouts.data(), (int)n_hops, p.node_capacity.empty() ? nullptr : p.node_capacity.data(), rng_seed,
                               stream_base, static_cast<const uint32_t*>(address(stream_offset)), flags, table_ptr, slots,
                               uniq.data_ptr<int32_t>(), p.cap_uniq, a[0].data(), a[1].data(), a[2].data(), transposed ? a[3].data() : nullptr,
                               transposed ? a[4].data() : nullptr, transposed ? a[5].data() : nullptr, counts.data_ptr<int32_t>(),
                               static_cast<int32_t*>(address(readback)), ws_ptr, (size_t)ws.numel(), stream);
        if (rc != FGL_OK) error = fgl_last_error();
    }
    TORCH_CHECK(rc == FGL_OK, "fastgl: ", error, " (error ", rc, ")");
    py::list ptrs, locals, globals, trans;
    for (size_t h = 0; h < n_hops; ++h) {
        ptrs.append(block_ptr[h]);
        locals.append(src_local[h]);
        globals.append(src_global[h]);
        if (t_ptr[h].defined()) trans.append(py::make_tuple(t_ptr[h], t_dst[h], t_edge[h]));
        else trans.append(py::none());
    }
    return py::make_tuple(uniq, ptrs, locals, globals, counts, trans);
}

// The arrays of a mini-batch cut to the sizes that came back (`c`: the call's counts): the unique list, and per hop, outermost first,
// (row offsets, local ids, graph ids or None, transposed arrays or None).
py::tuple trim(const torch::Tensor& uniq, const std::vector<torch::Tensor>& block_ptr, const std::vector<torch::Tensor>& src_local,
               const std::vector<Maybe>& src_global, const std::vector<c10::optional<std::vector<torch::Tensor>>>& transposed,
               const std::vector<int64_t>& c)
{
    const size_t n_hops = block_ptr.size();
    auto cut = [](const torch::Tensor& t, int64_t n) { return t.slice(0, 0, n); };
    py::list hops;
    for (size_t h = n_hops; h-- > 0;) {
        const int64_t n_dst = c[h], n_src = c[h + 1], n_e = c[n_hops + 1 + h];
        py::object global = py::none(), trans = py::none();
        if (src_global[h].has_value()) global = py::cast(cut(*src_global[h], n_e));
        if (transposed[h].has_value()) {
            const auto& t = *transposed[h];
            trans = py::make_tuple(cut(t[0], n_src + 1), cut(t[1], n_e), cut(t[2], n_e));
        }
        hops.append(py::make_tuple(cut(block_ptr[h], n_dst + 1), cut(src_local[h], n_e), global, trans));
    }
    return py::make_tuple(cut(uniq, c[n_hops]), hops);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    py::class_<Plan>(m, "Plan")
        .def(py::init([](std::vector<int32_t> fanouts, c10::optional<std::vector<int64_t>> node_capacity, std::vector<int64_t> cap_dst,
                         std::vector<int64_t> cap_edges, std::vector<int64_t> cap_src, int64_t cap_uniq, uint32_t transpose_mask) {
            return Plan{std::move(fanouts), node_capacity.has_value() ? std::move(*node_capacity) : std::vector<int64_t>(), std::move(cap_dst),
                        std::move(cap_edges), std::move(cap_src), cap_uniq, transpose_mask};
        }));
    m.def("sample_blocks", &sample_blocks);
    m.def("trim", &trim);
}
