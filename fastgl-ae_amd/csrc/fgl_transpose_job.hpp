// The transposed form of a sampled block, built inside the all-hops sampling call (fgl_sample_blocks) without a
// launch of its own wherever another launch of the call can carry the work.  (It is what turns the reference's
// atomic-scatter backward kernels, aggregate_acc_kernel.cu:467-517,554-596, into gathers; the reference builds
// nothing of the kind and the per-hop loop it runs instead is FusedMapSampler.py:72-107.)
//
// A counting sort by source node in five steps, each a grid-stride device function that any kernel of the
// right stream position can call on entry, before its own work:
//   zero        the per-column counters                    (the last launch of hop h-1; the call's first launch for h = 0)
//   rank        k = counter[col]++ for every edge, as its local source id becomes known
//                                                           (hop h's sampling and id-map launches: take_rank)
//   tile sums   per 2048 counters; the longest row         (hop h+1's sampling launch)
//   scan        counters -> offsets in place, the transposed row pointer
//                                                           (hop h+1's last id-map launch)
//   fill        t_dst[offset[col] + k] = row, t_edge[...] = edge     (hop h+2's sampling launch, or the call's closing launch)
// The last hop of a call has no hop after it: its closing steps are launches of their own.
// A carried step runs in workgroups of its own, appended to the carrying launch's grid (side_blocks of them,
// the last of the grid, see side_block): in front of the launch's own work it would lengthen the chain of
// memory latencies that a small hop's launch is (measured: 20 us per mini-batch, what the separate launches cost).
// Sizes that exist only on the device are read from the call's count array; every array is sized by the
// host-side bound.  `split` > 1 gives every column that many counters (entry e uses number e % split): returning
// atomics on one address complete one after the other, and a hub column of a large hop is mentioned thousands
// of times.
#pragma once
#include "fgl_common.hpp"
#include "fgl_kernels.hpp"

namespace fgl {

constexpr int kTjobTile = 2048;  // counters per scan tile

#if defined(__HIPCC__)

// rank of edge e within the transposed row of its local source id (-1: the edge has none)
__device__ __forceinline__ void take_rank(const TransposeRank& r, int64_t e, int32_t local)
{
    if (r.rank == nullptr) return;
    int32_t k = -1;
    if (local >= 0 && (int64_t)local < r.cols_max) k = atomicAdd(&r.cnt[(int64_t)local * r.split + (int)(e & (r.split - 1))], 1);
    r.rank[e] = k;
}

// This workgroup's index among the job's side workgroups -- the last side_blocks of the grid but side_first --
// or -1 if it is none of them.
__device__ __forceinline__ int side_block(const TransposeJob& j)
{
    const int64_t sb = (int64_t)gridDim.x - 1 - (int64_t)blockIdx.x - j.side_first;
    return (sb >= 0 && sb < j.side_blocks) ? (int)sb : -1;
}

__device__ __forceinline__ int64_t tjob_entries(const TransposeJob& j)
{
    return actual_count(j.cols_max, j.d_n_cols) * j.split + 1;  // one more: the total
}

template <int NT>
__device__ __forceinline__ void tjob_zero(const TransposeJob& j)
{
    if (j.cnt == nullptr) return;
    const int sb = side_block(j);
    if (sb < 0) return;
    const int64_t n = j.cols_max * j.split + 1;
    const int64_t stride = (int64_t)j.side_blocks * NT;
    for (int64_t i = (int64_t)sb * NT + threadIdx.x; i < n; i += stride) j.cnt[i] = 0;
}

template <int NT>
__device__ __forceinline__ void zero_job(const ZeroJob& j)
{
    if (j.n16 == 0) return;
    const int64_t sb = (int64_t)gridDim.x - 1 - (int64_t)blockIdx.x - j.side_first;
    if (sb < 0 || sb >= j.side_blocks) return;
    const uint4 z = make_uint4(0u, 0u, 0u, 0u);
    for (int64_t i = sb * NT + threadIdx.x; i < j.n16; i += (int64_t)j.side_blocks * NT) j.p[i] = z;
}

// ... and the longest row (if it holds more than FGL_SHORT_ROW_ENTRIES entries) into *longest, which starts at zero
template <int NT>
__device__ __forceinline__ void tjob_tile_sums(const TransposeJob& j)
{
    if (j.cnt == nullptr) return;
    __shared__ int smem[NT / kWave + 1];
    const int sb = side_block(j);
    if (sb < 0) return;  // (uniform over the workgroup: barriers below)
    const int64_t n = tjob_entries(j);
    const int64_t n_tiles = (n + kTjobTile - 1) / kTjobTile;
    for (int64_t tile = sb; tile < n_tiles; tile += j.side_blocks) {
        int v[kTjobTile / NT];
#pragma unroll
        for (int q = 0; q < kTjobTile / NT; ++q) {  // (all of the lane's loads in flight together)
            const int64_t i = tile * kTjobTile + (int64_t)q * NT + threadIdx.x;
            v[q] = (i < n - 1) ? j.cnt[i] : 0;  // (the last entry is the slot of the total: not a counter)
        }
        int s = 0, longest = 0;
#pragma unroll
        for (int q = 0; q < kTjobTile / NT; ++q) {
            s += v[q];
            int len = v[q];  // (a column's counters sit in neighbouring lanes)
            for (int d = 1; d < j.split; d <<= 1) len += __shfl_xor(len, d, kWave);
            longest = len > longest ? len : longest;
        }
        if (j.longest != nullptr && longest > FGL_SHORT_ROW_ENTRIES) atomicMax(j.longest, longest);
        const int total = block_sum_of_lanes<NT>(s, smem);
        if (threadIdx.x == 0) j.tile_sums[tile] = total;
    }
}

// counters -> exclusive prefix sums in place; t_ptr[c] = the prefix of column c's first counter
template <int NT>
__device__ __forceinline__ void tjob_scan(const TransposeJob& j)
{
    if (j.cnt == nullptr) return;
    constexpr int kItems = kTjobTile / NT;
    static_assert(kItems == 8 || kItems == 32, "tiles are dealt 8 (256 lanes) or 32 (64 lanes) counters per lane");
    __shared__ int smem[NT / kWave + 1];
    const int sb = side_block(j);
    if (sb < 0) return;  // (uniform over the workgroup: barriers below)
    const int64_t n = tjob_entries(j);
    const int64_t n_tiles = (n + kTjobTile - 1) / kTjobTile;
    const int split = j.split;
    for (int64_t tile = sb; tile < n_tiles; tile += j.side_blocks) {
        const int64_t base = tile * kTjobTile + (int64_t)threadIdx.x * kItems;
        int v[kItems];
        int s = 0;
#pragma unroll
        for (int q = 0; q < kItems; ++q) {
            v[q] = (base + q < n - 1) ? j.cnt[base + q] : 0;
            s += v[q];
        }
        const int before = block_sum_before<NT>(j.tile_sums, tile, smem);
        int total;
        int run = block_exclusive_scan<NT>(s, smem, &total) + before;
#pragma unroll
        for (int q = 0; q < kItems; ++q) {
            const int64_t i = base + q;
            if (i < n) {
                if (split > 1 || j.cnt != j.t_ptr) j.cnt[i] = run;
                if (split == 1) j.t_ptr[i] = run;
                else if ((i & (split - 1)) == 0) j.t_ptr[i / split] = run;
            }
            run += v[q];
        }
    }
}

// sixteen lanes per row of the block: its entries are read coalesced and scattered in parallel
template <int NT>
__device__ __forceinline__ void tjob_fill(const TransposeJob& j)
{
    if (j.cnt == nullptr) return;
    constexpr int kLanes = 16;
    const int sb = side_block(j);
    if (sb < 0) return;
    const int64_t n_rows = actual_count(j.rows_max, j.d_n_rows);
    const int64_t n_edges = actual_count(j.edges_max, j.d_n_edges);
    const int lane = (int)threadIdx.x % kLanes;
    const int split = j.split;
    const int64_t stride = (int64_t)j.side_blocks * (NT / kLanes);
    for (int64_t r = (int64_t)sb * (NT / kLanes) + (int)threadIdx.x / kLanes; r < n_rows; r += stride) {
        const int64_t a = j.block_ptr[r];
        int64_t b = j.block_ptr[r + 1];
        if (b > n_edges) b = n_edges;
        for (int64_t e = a + lane; e < b; e += kLanes) {
            const int32_t k = j.rank[e];
            if (k >= 0) {
                const int64_t pos = (int64_t)j.cnt[(int64_t)j.src_local[e] * split + (int)(e & (split - 1))] + k;
                if (pos < j.edges_max) {
                    j.t_dst[pos] = (int32_t)r;
                    if (j.t_edge) j.t_edge[pos] = (int32_t)e;
                }
            }
        }
    }
}

// ---- rows in a fixed order ------------------------------------------------------------------------------------
// The fill step leaves the entries of a transposed row in the order in which their atomics landed.  Sorting every
// row by the position of its entries in the block (t_edge; ascending positions = ascending destination rows,
// the order a stable counting sort gives) makes the transposed block, and with it the fp32 sums of every gather
// over it, the same from run to run.  Rows are short with few exceptions, so the work is dealt by length:
//   up to 8 entries     the row's lane sorts it in registers;
//   up to 64            the row's wave, one entry per lane, by shuffles;
//   longer rows         are listed by that pass and dealt out, one workgroup per row, by a second launch (hubs sit
//                       next to each other in the numbering: left to the workgroup that finds them they would queue
//                       up behind each other): up to kSortPiece entries in LDS;
//   beyond that         (a hub of a large mini-batch, or of a whole graph taken as one block) a workgroup per piece of kSortPiece
//                       entries: the second launch puts the pieces' keys in order, and a third one finds every key's place, which
//                       is its place in its piece plus the number of smaller keys in each of the others. (One workgroup per
//                       row, 4096 entries in LDS and then rounds of merging neighbours, took as many rounds as pieces, one behind the
//                       other: a row of 6000 / 20 000 / 100 000 entries sampled and put in order in 265 / 1042 / 14 633 us; now
//                       198 / 395 / 1548.  The five-hop mini-batch below: 66 -> 59 us, of which the third launch 27.)
// Keys are distinct (positions), or -- without t_edge -- destination rows, whose ties are interchangeable.
constexpr int kSortPiece = 2048;
constexpr int kSortBlock = 512;  // threads of a workgroup of the second and third launch
constexpr int kSortMax = 0x7FFFFFFF;

struct SortJobs {
    TransposeJob job[8];
    int32_t* long_rows;   // pairs (job + 8 * piece, row) of the rows left to the second launch
    int32_t* n_long;      // how many (zero when the first launch starts; may exceed long_max: then rows were dropped
    int64_t long_max;     //   from the list -- which its size, one per 65 entries, rules out)
};

__device__ __forceinline__ void sort_exchange(int& ka, int& va, int& kb, int& vb)
{
    if (kb < ka) {
        const int k = ka, v = va;
        ka = kb;
        va = vb;
        kb = k;
        vb = v;
    }
}

// the comparisons of a bitonic merge at distances below a wave, jj = first, first / 2, .. 1: one pair per lane, by shuffles
__device__ __forceinline__ void sort_lanes(int& k, int& v, int first, bool up)
{
    const int lane = lane_id();
    for (int jj = first; jj > 0; jj >>= 1) {
        const int ok = __shfl_xor(k, jj, kWave), ov = __shfl_xor(v, jj, kWave);
        const bool want_min = ((lane & jj) == 0) == up;
        if (want_min ? ok < k : k < ok) {  // (equal keys: both lanes keep theirs)
            k = ok;
            v = ov;
        }
    }
}

// bitonic sort of n (a power of two, 128 <= n <= kSortPiece) pairs in LDS by the whole workgroup.  What bounds it is the chain of
// steps (66 for 2048 pairs), each a pass over LDS and a barrier: the 51 at distances below a wave are done in registers, a wave per 64
// neighbours, which leaves 15 barriers of that kind and 6 around the register passes.  The long rows of a five-hop mini-batch (1000 seeds,
// 2.4 M nodes), with 512 threads a piece instead of 256: 98 -> 67 us (1024 threads: 65, and half as many pieces at a time).
template <int NT>
__device__ __forceinline__ void sort_lds(int* s_key, int* s_val, int n)
{
    for (int i = threadIdx.x; i < n; i += NT) {  // (n and NT are multiples of a wave)
        int k = s_key[i], v = s_val[i];
        for (int run = 2; run <= kWave; run <<= 1) sort_lanes(k, v, run >> 1, (i & run) == 0);
        s_key[i] = k;
        s_val[i] = v;
    }
    __syncthreads();
    for (int k = 2 * kWave; k <= n; k <<= 1) {
        for (int jj = k >> 1; jj >= kWave; jj >>= 1) {
            for (int t = threadIdx.x; t < n / 2; t += NT) {
                const int i = 2 * t - (t & (jj - 1));  // the lower index of the t-th pair at distance jj
                const int o = i + jj;
                const bool up = (i & k) == 0 || k == n;  // (the last merge is ascending throughout)
                int ka = s_key[i], va = s_val[i], kb = s_key[o], vb = s_val[o];
                if (up ? kb < ka : ka < kb) {
                    s_key[i] = kb;
                    s_val[i] = vb;
                    s_key[o] = ka;
                    s_val[o] = va;
                }
            }
            __syncthreads();
        }
        for (int i = threadIdx.x; i < n; i += NT) {
            int key = s_key[i], val = s_val[i];
            sort_lanes(key, val, kWave / 2, (i & k) == 0 || k == n);
            s_key[i] = key;
            s_val[i] = val;
        }
        __syncthreads();
    }
}

template <int NT>
__device__ __forceinline__ void sort_load(int* s_key, int* s_val, const int32_t* key, const int32_t* val, int64_t a, int len, int n)
{
    for (int i = threadIdx.x; i < n; i += NT) {
        s_key[i] = i < len ? key[a + i] : kSortMax;
        s_val[i] = (val != nullptr && i < len) ? val[a + i] : 0;
    }
}

template <int NT>
__device__ __forceinline__ void sort_store(const int* s_key, const int* s_val, int32_t* key, int32_t* val, int64_t a, int len)
{
    for (int i = threadIdx.x; i < len; i += NT) {
        key[a + i] = s_key[i];
        if (val != nullptr) val[a + i] = s_val[i];
    }
}

template <int NT>
__device__ __forceinline__ void tjob_sort_rows(const SortJobs& jobs, int job_index)
{
    const TransposeJob& j = jobs.job[job_index];
    if (j.t_ptr == nullptr) return;
    int32_t* key = j.t_edge ? j.t_edge : j.t_dst;
    int32_t* val = j.t_edge ? j.t_dst : nullptr;
    const int64_t n_cols = actual_count(j.cols_max, j.d_n_cols);
    const int64_t n_edges = actual_count(j.edges_max, j.d_n_edges);
    const int lane = lane_id();
    // Neighbouring rows go to different waves (row r to wave r mod the number of waves): the long rows of a block
    // sit next to each other -- hubs are met early and numbered early -- and a wave takes its rows of 9..64 entries
    // one after the other.
    const int64_t n_waves = (int64_t)gridDim.x * (NT / kWave);
    const int64_t wave = (int64_t)blockIdx.x * (NT / kWave) + threadIdx.x / kWave;
    for (int64_t first = 0; first < n_cols; first += n_waves * kWave) {  // (uniform over the launch)
        const int64_t c = first + wave + n_waves * lane;
        int64_t a = 0, b = 0;
        if (c < n_cols) {
            a = j.t_ptr[c];
            b = j.t_ptr[c + 1];
            if (b > n_edges) b = n_edges;
            if (a > b) a = b;
        }
        const int64_t len = b - a;
        if (len >= 2 && len <= 8) {  // in registers: a sorting network for eight
            int k[8], v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                k[i] = i < len ? key[a + i] : kSortMax;
                v[i] = (val != nullptr && i < len) ? val[a + i] : 0;
            }
#define FGL_CX(x, y) sort_exchange(k[x], v[x], k[y], v[y])
            FGL_CX(0, 1); FGL_CX(2, 3); FGL_CX(4, 5); FGL_CX(6, 7);
            FGL_CX(0, 2); FGL_CX(1, 3); FGL_CX(4, 6); FGL_CX(5, 7);
            FGL_CX(1, 2); FGL_CX(5, 6); FGL_CX(0, 4); FGL_CX(3, 7);
            FGL_CX(1, 5); FGL_CX(2, 6);
            FGL_CX(1, 4); FGL_CX(3, 6);
            FGL_CX(2, 4); FGL_CX(3, 5);
            FGL_CX(3, 4);
#undef FGL_CX
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (i < len) {
                    key[a + i] = k[i];
                    if (val != nullptr) val[a + i] = v[i];
                }
        }
        // rows of 9..64 entries: the wave takes them one after the other, an entry per lane
        unsigned long long todo = __ballot(len > 8 && len <= kWave);
        while (todo != 0) {
            const int r = __ffsll((long long)todo) - 1;
            todo &= todo - 1;
            const int64_t ra = __shfl(a, r, kWave);
            const int rl = (int)__shfl(len, r, kWave);
            int kk = lane < rl ? key[ra + lane] : kSortMax;
            int vv = (val != nullptr && lane < rl) ? val[ra + lane] : 0;
#pragma unroll
            for (int k2 = 2; k2 <= kWave; k2 <<= 1) {
#pragma unroll
                for (int jj = k2 >> 1; jj > 0; jj >>= 1) {
                    const int ok = __shfl_xor(kk, jj, kWave);
                    const int ov = __shfl_xor(vv, jj, kWave);
                    const bool up = (lane & k2) == 0;
                    const bool lower = (lane & jj) == 0;
                    const bool take = (lower == up) ? (ok < kk) : (ok > kk);
                    if (take) {
                        kk = ok;
                        vv = ov;
                    }
                }
            }
            if (lane < rl) {
                key[ra + lane] = kk;
                if (val != nullptr) val[ra + lane] = vv;
            }
        }
        // longer rows: listed for the second launch, piece by piece
        if (len > kWave) {
            const int pieces = (int)((len + kSortPiece - 1) / kSortPiece);
            const int64_t at = atomicAdd(jobs.n_long, pieces);
            for (int p = 0; p < pieces; ++p) {
                if (at + p >= jobs.long_max) break;
                jobs.long_rows[2 * (at + p)] = job_index + 8 * p;
                jobs.long_rows[2 * (at + p) + 1] = (int32_t)c;
            }
        }
    }
}

// the piece that entry q of the list names: its first entry and its length, and those of its row
struct SortPiece {
    int64_t row_a, row_len, a;
    int len;
};
__device__ __forceinline__ SortPiece sort_piece(const SortJobs& jobs, const TransposeJob& j, int64_t q)
{
    const int64_t c = jobs.long_rows[2 * q + 1];
    const int64_t n_edges = actual_count(j.edges_max, j.d_n_edges);
    int64_t a = j.t_ptr[c], b = j.t_ptr[c + 1];
    if (b > n_edges) b = n_edges;
    if (a > b) a = b;
    SortPiece p;
    p.row_a = a;
    p.row_len = b - a;
    const int64_t from = (int64_t)(jobs.long_rows[2 * q] >> 3) * kSortPiece;
    p.a = a + from;
    const int64_t left = b - p.a;
    p.len = left <= 0 ? 0 : left < kSortPiece ? (int)left : kSortPiece;
    return p;
}

// second launch: rows of one piece in place; the keys of the others' pieces, in order, to where the ranks were
template <int NT>
__device__ __forceinline__ void tjob_sort_long_rows(const SortJobs& jobs, int* s_key, int* s_val)
{
    int64_t total = *jobs.n_long;
    if (total > jobs.long_max) total = jobs.long_max;
    for (int64_t q = blockIdx.x; q < total; q += gridDim.x) {
        const TransposeJob& j = jobs.job[jobs.long_rows[2 * q] & 7];
        const SortPiece p = sort_piece(jobs, j, q);
        const bool alone = p.row_len <= kSortPiece;
        int32_t* key = j.t_edge ? j.t_edge : j.t_dst;
        int32_t* val = alone && j.t_edge ? j.t_dst : nullptr;
        int n = 128;
        while (n < p.len) n <<= 1;
        sort_load<NT>(s_key, s_val, key, val, p.a, p.len, n);
        __syncthreads();
        sort_lds<NT>(s_key, s_val, n);
        sort_store<NT>(s_key, s_val, alone ? key : j.rank, val, p.a, p.len);
        __syncthreads();
    }
}

// third launch: the keys of rows of several pieces to their places; an entry's destination row is the block's row that holds its
// position, looked up again (the pieces moved without it)
template <int NT>
__device__ __forceinline__ void tjob_merge_long_rows(const SortJobs& jobs, int* s_key)
{
    constexpr int kItems = kSortPiece / NT;
    int64_t total = *jobs.n_long;
    if (total > jobs.long_max) total = jobs.long_max;
    for (int64_t q = blockIdx.x; q < total; q += gridDim.x) {
        const TransposeJob& j = jobs.job[jobs.long_rows[2 * q] & 7];
        const SortPiece p = sort_piece(jobs, j, q);
        if (p.row_len <= kSortPiece) continue;  // (uniform over the workgroup)
        int key[kItems];
        int64_t at[kItems];
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int i = (int)threadIdx.x + u * NT;
            key[u] = i < p.len ? j.rank[p.a + i] : kSortMax;
            at[u] = p.row_a + i;
        }
        for (int64_t o = p.row_a; o < p.row_a + p.row_len; o += kSortPiece) {
            if (o == p.a) continue;
            const int64_t left = p.row_a + p.row_len - o;
            const int len = left < kSortPiece ? (int)left : kSortPiece;
            for (int i = threadIdx.x; i < len; i += NT) s_key[i] = j.rank[o + i];
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kItems; ++u) {
                int lo = 0, hi = len;  // (equal keys -- only without positions -- stay in the order of their pieces)
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (o < p.a ? s_key[mid] <= key[u] : s_key[mid] < key[u]) lo = mid + 1; else hi = mid;
                }
                at[u] += lo;
            }
            __syncthreads();
        }
        const int64_t n_rows = actual_count(j.rows_max, j.d_n_rows);
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            if ((int)threadIdx.x + u * NT >= p.len) continue;
            if (j.t_edge == nullptr) {
                j.t_dst[at[u]] = key[u];
                continue;
            }
            j.t_edge[at[u]] = key[u];
            int64_t lo = 0, hi = n_rows;  // block_ptr[lo] <= key < block_ptr[hi]
            while (hi - lo > 1) {
                const int64_t mid = (lo + hi) >> 1;
                if (j.block_ptr[mid] <= key[u]) lo = mid; else hi = mid;
            }
            j.t_dst[at[u]] = (int32_t)lo;
        }
    }
}

#endif  // __HIPCC__

}  // namespace fgl
