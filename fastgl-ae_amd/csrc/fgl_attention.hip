// Attention coefficients of a GAT layer over a block CSR: for every destination row r and head h
//   s(e)     = leaky_relu(el[indices[e], h] + er[r, h])          e in [indptr[r], indptr[r+1])
//   alpha(e) = exp(s(e) - max_e' s(e')) / sum_e' exp(s(e') - max)
// -- what the reference gets from three DGL calls (apply_edges(u_add_v), leaky_relu,
// edge_softmax; GraphConv.py:265-272) and what a torch restatement spends ten launches over
// [n_entries, n_heads] on.  The result feeds FGL_AGG_EDGE as its per-entry weights.
//
// One lane per (row, head), the heads of a row in neighbouring lanes (they read the same
// neighbour id and 4 * n_heads contiguous bytes of el).  Two passes over the row's entries: a
// running maximum with a rescaled running sum, then the normalised values; the scores are
// recomputed in the second pass (the reads hit in cache) rather than kept.  Sampled blocks hold at
// most `fanout` entries per row; a hub row of an unsampled block is walked by its one lane.
#include "fgl_common.hpp"
#include "fgl_kernels.hpp"

namespace fgl {

__global__ __launch_bounds__(kBlock) void edge_softmax_kernel(const int32_t* __restrict__ indptr,
                                                              const int32_t* __restrict__ indices, int64_t n_rows_max,
                                                              const int32_t* __restrict__ d_n_rows,
                                                              const float* __restrict__ el, const float* __restrict__ er,
                                                              int n_heads, float negative_slope, float* __restrict__ alpha)
{
    const int64_t n_rows = actual_count(n_rows_max, d_n_rows);
    const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    const int64_t row = t / n_heads;
    if (row >= n_rows) return;
    const int h = (int)(t - row * n_heads);
    const int a = indptr[row], b = indptr[row + 1];
    const float r = er[row * n_heads + h];
    float top = -INFINITY, sum = 0.0f;
    for (int e = a; e < b; ++e) {
        float s = el[(int64_t)indices[e] * n_heads + h] + r;
        s = s > 0.0f ? s : negative_slope * s;
        if (s > top) {
            sum = sum * expf(top - s) + 1.0f;  // (first entry: 0 * exp(-inf) + 1)
            top = s;
        } else {
            sum += expf(s - top);
        }
    }
    const float inv = 1.0f / sum;
    for (int e = a; e < b; ++e) {
        float s = el[(int64_t)indices[e] * n_heads + h] + r;
        s = s > 0.0f ? s : negative_slope * s;
        alpha[(int64_t)e * n_heads + h] = expf(s - top) * inv;
    }
}

// el[i, h] = sum_f x[i, h, f] * attn_l[h, f] for all rows and er[i, h] likewise with attn_r for the first n_er rows, from one
// pass over x, which is what bounds it.  Sixteen lanes take one head of four rows: the heads of a row are neighbouring
// lane groups, so a wave's load of 64-column heads is one kilobyte of a row, four rows in flight; the sums over the lanes are a
// fixed-order __shfl_xor tree.
// Measured against the two products and two sums of torch that it replaces, three layers of a 1000-seed GAT step (4 heads of
// 64 columns, 107 K rows in the first): 255 -> 30 us.
constexpr int kScoreLanes = 16, kScoreRows = 4;

template <int VEC>
__global__ __launch_bounds__(kBlock) void head_scores_kernel(const float* __restrict__ x, int64_t ldx, int64_t n, int64_t n_er, int n_heads, int width,
                                                             const float* __restrict__ attn_l, const float* __restrict__ attn_r,
                                                             float* __restrict__ el, float* __restrict__ er)
{
    typedef float Vec __attribute__((ext_vector_type(VEC), aligned(4)));
    const int64_t group = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / kScoreLanes;
    const int lane = (int)(threadIdx.x % kScoreLanes);
    const int64_t row0 = group / n_heads * kScoreRows;
    const int h = (int)(group % n_heads);
    if (row0 >= n) return;  // (the same for all lanes of a group)
    const int64_t last = n - 1;
    const float* p[kScoreRows];
    float l[kScoreRows], r[kScoreRows];
#pragma unroll
    for (int i = 0; i < kScoreRows; ++i) {
        p[i] = x + (row0 + i < n ? row0 + i : last) * ldx + (int64_t)h * width;
        l[i] = r[i] = 0.0f;
    }
    const float *wl = attn_l + (int64_t)h * width, *wr = attn_r + (int64_t)h * width;
    for (int f = lane * VEC; f < width; f += kScoreLanes * VEC) {
        Vec v[kScoreRows];
#pragma unroll
        for (int i = 0; i < kScoreRows; ++i) v[i] = *reinterpret_cast<const Vec*>(p[i] + f);
        const Vec a = *reinterpret_cast<const Vec*>(wl + f), b = *reinterpret_cast<const Vec*>(wr + f);
#pragma unroll
        for (int i = 0; i < kScoreRows; ++i)
#pragma unroll
            for (int c = 0; c < VEC; ++c) {
                l[i] = fmaf(v[i][c], a[c], l[i]);
                r[i] = fmaf(v[i][c], b[c], r[i]);
            }
    }
#pragma unroll
    for (int d = kScoreLanes / 2; d >= 1; d >>= 1)
#pragma unroll
        for (int i = 0; i < kScoreRows; ++i) {
            l[i] += __shfl_xor(l[i], d, kScoreLanes);
            r[i] += __shfl_xor(r[i], d, kScoreLanes);
        }
#pragma unroll
    for (int i = 0; i < kScoreRows; ++i) {
        if (lane != i || row0 + i >= n) continue;
        el[(row0 + i) * n_heads + h] = l[i];
        if (row0 + i < n_er) er[(row0 + i) * n_heads + h] = r[i];
    }
}

}  // namespace fgl

using namespace fgl;

FGL_EXPORT int fgl_edge_softmax(const int32_t* d_indptr, const int32_t* d_indices, int64_t n_rows_max,
                                const int32_t* d_n_rows, const float* d_el, const float* d_er, int n_heads,
                                float negative_slope, float* d_alpha, void* stream)
{
    FGL_REQUIRE(n_rows_max >= 0, "edge_softmax: negative row count");
    FGL_REQUIRE(n_heads >= 1 && n_heads <= 1024, "edge_softmax: head count %d outside [1, 1024]", n_heads);
    if (n_rows_max == 0) return FGL_OK;
    FGL_REQUIRE(d_indptr && d_indices && d_el && d_er && d_alpha, "edge_softmax: null pointer");
    const int64_t blocks = ceil_div(n_rows_max * n_heads, kBlock);
    FGL_REQUIRE(blocks <= 0x7FFFFFFF, "edge_softmax: grid too large");
    hipLaunchKernelGGL(edge_softmax_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, as_stream(stream), d_indptr, d_indices,
                       n_rows_max, d_n_rows, d_el, d_er, n_heads, negative_slope, d_alpha);
    FGL_CHECK_LAUNCH("edge_softmax_kernel");
    return FGL_OK;
}

FGL_EXPORT int fgl_head_scores(const float* d_x, int64_t ldx, int64_t n_rows, int64_t n_er, int n_heads, int width, const float* d_attn_l,
                               const float* d_attn_r, float* d_el, float* d_er, void* stream)
{
    FGL_REQUIRE(n_rows >= 0 && n_er >= 0 && n_er <= n_rows, "head_scores: row counts %lld, %lld", (long long)n_rows, (long long)n_er);
    FGL_REQUIRE(n_heads >= 1 && width >= 1, "head_scores: %d heads of %d columns", n_heads, width);
    FGL_REQUIRE(ldx >= (int64_t)n_heads * width, "head_scores: row stride smaller than the row length");
    if (n_rows == 0) return FGL_OK;
    FGL_REQUIRE(d_x && d_attn_l && d_attn_r && d_el && (d_er || n_er == 0), "head_scores: null pointer");
    const int64_t blocks = ceil_div(ceil_div(n_rows, kScoreRows) * n_heads * kScoreLanes, kBlock);
    FGL_REQUIRE(blocks <= 0x7FFFFFFF, "head_scores: grid too large");
    const dim3 grid((unsigned)blocks), block(kBlock);
    if (width % 4 == 0)
        hipLaunchKernelGGL((head_scores_kernel<4>), grid, block, 0, as_stream(stream), d_x, ldx, n_rows, n_er, n_heads, width, d_attn_l, d_attn_r, d_el, d_er);
    else
        hipLaunchKernelGGL((head_scores_kernel<1>), grid, block, 0, as_stream(stream), d_x, ldx, n_rows, n_er, n_heads, width, d_attn_l, d_attn_r, d_el, d_er);
    FGL_CHECK_LAUNCH("head_scores_kernel");
    return FGL_OK;
}
