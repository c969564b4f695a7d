// Counting and block transpose for large inputs, without an atomic per entry in device memory (stands in for the reference's
// cal_deg, cuda_operators/utilis.cu:43-79, and -- as the transposed block that its backward kernels are gathers over -- for
// its atomic scatter, aggregate_acc_kernel.cu:467-517,554-596).
//
// What bounds the plain form: every entry is one atomic on its id's counter.  The chip retires about 24 G of them a second
// on random addresses, but updates of one address complete one after the other, some 90 ns each with a returned value, and
// graphs have hubs: one id mentioned 85 K times holds a count of 54 M ids for 8.5 ms whatever the rest does.
//
// Two forms, by size:
//
// (1) ids against ranges (count_ranges_kernel, up to a few million ids over half a million counters): a workgroup owns a range
//     of 16384 counters in LDS and reads a slice of the ids, counting those in its range; the slices' counts are stored and
//     added by a second launch.  Every id is read once per range -- from cache -- and no counter is shared between workgroups.
//     (1.2 M ids of a sampled block over 310 K counters: 66 -> 23 us.)
//
// (2) partition, then count (bucket_*): the entries are dealt into buckets of neighbouring columns (2^11 .. 2^13 wide) with one
//     pass -- per tile of entries a histogram over the buckets in LDS, one scan over (bucket, tile), and a pass
//     that puts the tile in order in LDS and stores every bucket's entries at its place -- and then counted bucket by bucket in
//     LDS, a workgroup per segment of a bucket.  The transpose goes on from there: a segment learns its place in each of its
//     columns from the add that delivers its counts (one atomic per segment and column), the counts are scanned into offsets,
//     and the segment's entries are put in order by column in LDS and stored as runs.
//     Within a bucket a column is 16 bits.  Traffic: 2 reads of the ids, 2 writes and reads of the rows, 1 write and 2 reads of
//     half the columns.
//     (54 M entries of a 2.4 M-node graph, hubs of 85 K, us: counts, with an atomic per entry 5900 / 13200 -- unordered / sorted
//     ids --, with 4-byte stores all over the buckets 499 / 674, now 276 / 180; transpose 24700, 1550, now 700.)
#include "fgl_common.hpp"
#include "fgl_kernels.hpp"
#include "fgl_tile_rows.hpp"

namespace fgl {

// ---- (1) ids against ranges -------------------------------------------------------------------------------------
constexpr int kRangeCounters = 16384;  // 64 KiB of LDS: two workgroups per CU
constexpr int kRangeBlock = 1024;

__global__ __launch_bounds__(kRangeBlock) void count_ranges_kernel(const int32_t* __restrict__ ids, int64_t n_max,
                                                                   const int32_t* __restrict__ d_n, int64_t per_slice,
                                                                   int64_t n_counters, int32_t* __restrict__ partial)
{
    __shared__ int s_cnt[kRangeCounters];
    for (int i = (int)threadIdx.x; i < kRangeCounters; i += kRangeBlock) s_cnt[i] = 0;
    __syncthreads();
    const int64_t n = actual_count(n_max, d_n);
    const int64_t first = (int64_t)blockIdx.y * per_slice;
    const int64_t last = first + per_slice < n ? first + per_slice : n;
    const int64_t base = (int64_t)blockIdx.x * kRangeCounters;
    const int width = n_counters - base < kRangeCounters ? (int)(n_counters - base) : kRangeCounters;
    constexpr int kInFlight = 8;
    int64_t i = first + threadIdx.x;
    for (; i + (kInFlight - 1) * kRangeBlock < last; i += kInFlight * kRangeBlock) {
        int32_t id[kInFlight];
#pragma unroll
        for (int j = 0; j < kInFlight; ++j) id[j] = ids[i + (int64_t)j * kRangeBlock];
#pragma unroll
        for (int j = 0; j < kInFlight; ++j) {
            const int64_t at = (int64_t)id[j] - base;
            if (at >= 0 && at < width) atomicAdd(&s_cnt[at], 1);
        }
    }
    for (; i < last; i += kRangeBlock) {
        const int64_t at = (int64_t)ids[i] - base;
        if (at >= 0 && at < width) atomicAdd(&s_cnt[at], 1);
    }
    __syncthreads();
    for (int c = (int)threadIdx.x; c < width; c += kRangeBlock) partial[(int64_t)blockIdx.y * n_counters + base + c] = s_cnt[c];
}

__global__ __launch_bounds__(kBlock) void count_ranges_sum_kernel(const int32_t* __restrict__ partial, int slices, int64_t n_counters,
                                                                  int32_t* __restrict__ out)
{
    const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c >= n_counters) return;
    int s = 0;
    int q = 0;
    for (; q + 4 <= slices; q += 4) {
        const int v0 = partial[q * n_counters + c], v1 = partial[(q + 1) * n_counters + c];
        const int v2 = partial[(q + 2) * n_counters + c], v3 = partial[(q + 3) * n_counters + c];
        s += (v0 + v1) + (v2 + v3);
    }
    for (; q < slices; ++q) s += partial[q * n_counters + c];
    out[c] = s;
}

// ---- (2) buckets ------------------------------------------------------------------------------------------------
constexpr int kBucketBlock = 512;
constexpr int kBucketItems = 16;  // entries per lane
constexpr int kBucketTile = kBucketBlock * kBucketItems;  // entries that are put in order in LDS together
constexpr int kMaxBuckets = 2048;
constexpr int kMinWidthLog = 11, kMaxWidthLog = 13;
constexpr int kSegment = 32768, kMinSegment = 8192;  // entries per workgroup of the passes over buckets: BucketArgs::segment, between these

struct BucketArgs {
    const int32_t* ids;          // column of every entry
    int64_t n_max;               // entries: at most this many, *d_n or indptr[n_rows] of them
    const int32_t* d_n;
    const int32_t* indptr;       // transpose only: rows of the entries
    int64_t n_rows;
    int64_t n_cols;
    int width_log, buckets, segment;
    int64_t tiles;               // of kBucketTile entries
    int32_t* hist;               // [bucket][tile] counts, then their prefix sums (+ 1 entry: the total)
    int32_t* tile_row;           // [tile] the row that holds the tile's first entry
    int32_t* direct;             // [tile] counting only: 1 where bucket_hist_kernel has counted the tile's entries already
    uint16_t* b_col;             // entries by bucket: column within the bucket, row, position in ids
    int32_t* b_row;
    int32_t* b_edge;
    int32_t* segments;           // [0] = how many, then per segment {bucket, first entry, entries}
    int32_t* seg_base;           // [segment][2^width_log] a segment's first place in each of its columns
    int32_t* counts;             // n_cols
    int32_t* longest;            // (may be null) zeroed by the first launch
    int32_t* t_indices;
    int32_t* t_edge;
};

__device__ __forceinline__ int64_t bucket_entries(const BucketArgs& g)
{
    if (g.indptr == nullptr) return actual_count(g.n_max, g.d_n);
    const int64_t n = g.n_rows > 0 ? (int64_t)g.indptr[g.n_rows] : 0;
    return n < g.n_max ? n : g.n_max;
}

// Workgroup -> tile (the grid is a multiple of eight): every XCD takes a contiguous eighth, in order.  Workgroups go to the
// XCDs in turn and each XCD has its own L2: neighbouring tiles write next to each other (a histogram's row, a bucket's next
// entries), and only in one L2 do their pieces become whole lines.
__device__ __forceinline__ int64_t xcd_tile(int64_t n)
{
    const int64_t per = (n + 7) / 8;
    const int64_t i = (int64_t)(blockIdx.x / 8), at = (int64_t)(blockIdx.x % 8) * per + i;
    return i < per && at < n ? at : -1;
}

// counters to zero; the row of every tile's first entry (each row names the tiles that begin inside it)
__global__ __launch_bounds__(kBlock) void bucket_init_kernel(const BucketArgs g)
{
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    const int64_t first = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (g.longest != nullptr && first == 0) *g.longest = 0;
    for (int64_t i = first; i < g.n_cols; i += stride) g.counts[i] = 0;
    if (g.indptr == nullptr) return;
    for (int64_t r = first; r < g.n_rows; r += stride) mark_tile_rows<kBucketTile>(g.indptr, r, g.tiles, g.tile_row);
}

// the bucket of each of a lane's neighbouring entries (-1: no such entry, or no such column)
__device__ __forceinline__ void load_columns(const BucketArgs& g, int64_t first, int64_t n, int32_t (&c)[kBucketItems])
{
    typedef int32_t I4 __attribute__((ext_vector_type(4), aligned(4)));
    if (first + kBucketItems <= n) {
#pragma unroll
        for (int q = 0; q < kBucketItems / 4; ++q) {
            const I4 v = *reinterpret_cast<const I4*>(g.ids + first + 4 * q);
#pragma unroll
            for (int j = 0; j < 4; ++j) c[4 * q + j] = v[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < kBucketItems; ++j) c[j] = first + j < n ? g.ids[first + j] : -1;
    }
#pragma unroll
    for (int j = 0; j < kBucketItems; ++j)
        if (c[j] >= g.n_cols) c[j] = -1;
}

// A tile's entries by bucket.  (A lane's entries are neighbours, and equal ones are counted together: sorted ids -- a CSR's
// rows -- would otherwise be 64 updates of one counter at a time, one after the other.)
// DIRECT (counting only): a tile of an input in order, in runs of equal ids -- the destinations of an edge list -- is counted
// here, one atomic a run in device memory, and the launches behind pass it by; what two tiles share of a hub is one atomic each.
// In order is more than the tile's own ids: device memory does not take updates of the same few counters from all over the chip.
// So the first ids of the input's 64 parts of neighbouring tiles have to ascend, and those of 64 tiles of the tile's own part (all of
// them up to 33 M ids), and the tile's ids, from the tile before on, to lie between those of its part and the next one: a counter is
// touched by neighbouring tiles, most of them one XCD's, or by parts that hold one id.
// Whole counts, us, by buckets alone / with it: 54 M destinations of an R-MAT graph of 2.4 M nodes 272 / 179, sorted uniform ids,
// 22 a run, 270 / 180, 11 a run 277 / 251, in no order 280 / 280; 20 M over 900 K, sorted 82 / 70; 5 M over 500 K, sorted, 46 / 35,
// over 600 K, eight a run, 42 / 39, in no order 37.4 / 38.3.  Sorted stretches, which only cost the look: 54 M in stretches of two tiles
// over 500 ids 254 / 264, of such that begin anew for each 64th part 201 / 210.
// kDirectRun of 5: sorted uniform ids of five a run 348, six 341 where 6 takes 310 and 292; of 8: 310 and 280, but skewed sorted ids (u^4
// of 2.5 M, 22 a run) 256 where 6 takes 213 (buckets 274).  Without the parts, stretches of two tiles over 500 ids took 879; without the
// tiles of a part, such that begin anew for each part, five a run, 510; when the tile's first wave alone was looked at, for runs of four,
// fives of two ids in turn 122477, tiles in order up to their eighth 1857.
constexpr int kDirectRun = 6;

template <bool DIRECT>
__global__ __launch_bounds__(kBucketBlock) void bucket_hist_kernel(const BucketArgs g)
{
    __shared__ int s_cnt[kMaxBuckets];
    const int64_t n = bucket_entries(g);
    const int64_t tile = xcd_tile(g.tiles);
    if (tile < 0) return;
    const int tid = (int)threadIdx.x;
    for (int b = tid; b < g.buckets; b += kBucketBlock) s_cnt[b] = 0;
    int32_t c[kBucketItems];
    int32_t before = -1;  // the last entry of the tile before
    if (DIRECT && tid == 0 && tile > 0 && tile * kBucketTile <= n) before = g.ids[tile * kBucketTile - 1];
    load_columns(g, tile * kBucketTile + (int64_t)tid * kBucketItems, n, c);
    bool direct = false;
    if constexpr (DIRECT) {
        constexpr int kWaves = kBucketBlock / kWave;
        __shared__ int s_direct, s_most, s_runs, s_last[kBucketBlock], s_first[kWaves];
        const int lane = lane_id(), wave = tid / kWave;
        // one wave looks at its 1024 entries, for all: what the others would see costs an input in no order 2 % of the whole
        // count (the runs that begin in the wave, and whether the lane's ids ascend)
        // (what lies past the end goes with the ids before it: the last tile alone in buckets kept the launches behind waiting, 8.9 M sorted
        // ids over 176 counters 31 us where they take 24)
        const int64_t behind = n - (tile * kBucketTile + (int64_t)tid * kBucketItems);
        const int left = behind < 0 ? 0 : behind < kBucketItems ? (int)behind : kBucketItems;
        auto look = [&](int last, bool& ascends) {
            int begin = c[0] != last;
            ascends = c[0] >= last || left == 0;
#pragma unroll
            for (int j = 1; j < kBucketItems; ++j) {
                begin += c[j] != c[j - 1];
                ascends &= c[j] >= c[j - 1] || j >= left;
            }
            int runs = 0;
#pragma unroll
            for (int b = 0; b < 5; ++b) runs += __popcll(__ballot(begin >> b & 1)) << b;
            return runs;
        };
        bool ascends;
        if (tid < kWave) {
            const int last = __shfl_up(c[kBucketItems - 1], 1, kWave);
            const int runs = look(tid > 0 ? last : before < g.n_cols ? before : -1, ascends);
            bool may_be = __all(ascends) && runs <= kWave * kBucketItems / kDirectRun;
            int most = INT32_MAX;
            if (may_be) {  // (uniform) the first ids of the input's parts, a lane each
                const int per = (int)((g.tiles + kWave - 1) / kWave), part = (int)tile / per;
                const int64_t at = (int64_t)lane * per * kBucketTile;
                int begin = INT32_MAX;
                if (at < n) {
                    begin = g.ids[at];
                    if (begin >= g.n_cols) begin = -1;
                }
                int next = __shfl_down(begin, 1, kWave);
                if (lane == kWave - 1) next = INT32_MAX;
                most = __shfl(next, part, kWave);
                may_be = __all(begin <= next) && __all(c[0] >= __shfl(begin, part, kWave) || left == 0);
                if (may_be) {  // and the first ids of 64 tiles of its part
                    const int64_t from = ((int64_t)part * per + (int64_t)lane * per / kWave) * kBucketTile;
                    int id = INT32_MAX;
                    if (from < n) {
                        id = g.ids[from];
                        if (id >= g.n_cols) id = -1;
                    }
                    int after = __shfl_down(id, 1, kWave);
                    if (lane == kWave - 1) after = most;
                    may_be = __all(id <= after);
                }
            }
            if (tid == 0) {
                s_direct = may_be;
                s_most = most;
                s_runs = 0;
            }
        }
        __syncthreads();
        direct = s_direct != 0;
        if (direct) {  // (the whole workgroup): now all of it
            s_last[tid] = c[kBucketItems - 1];
            __syncthreads();
            const int runs = look(tid > 0 ? s_last[tid - 1] : -1, ascends);
            if (lane == 0) atomicAdd(&s_runs, runs);
            direct = __syncthreads_and(ascends && c[kBucketItems - 1] <= s_most) != 0 && s_runs <= kBucketTile / kDirectRun;
        }
        if (tid == 0) g.direct[tile] = direct;
        if (direct) {
            uint32_t heads = 0;  // where runs begin: bit j for the lane's entry j
#pragma unroll
            for (int j = 1; j < kBucketItems; ++j) heads |= c[j] != c[j - 1] ? 1u << j : 0u;
            if (tid == 0 || c[0] != s_last[tid - 1]) heads |= 1u;
            // the first of them, as a place in the tile, in this lane or behind it in the wave
            int first = heads != 0 ? tid * kBucketItems + __ffs((int)heads) - 1 : kBucketTile;
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
                const int t = __shfl_down(first, d, kWave);
                if (lane + d < kWave && t < first) first = t;
            }
            if (lane == 0) s_first[wave] = first;
            __syncthreads();
            int next = __shfl_down(first, 1, kWave);
            if (lane == kWave - 1) next = kBucketTile;
#pragma unroll
            for (int w = 0; w < kWaves; ++w)
                if (w > wave && s_first[w] < next) next = s_first[w];
#pragma unroll
            for (int j = kBucketItems - 1; j >= 0; --j) {
                if ((heads >> j & 1) == 0) continue;
                const int at = tid * kBucketItems + j;
                if (c[j] >= 0) atomicAdd(&g.counts[c[j]], next - at);
                next = at;
            }
        }
    } else {
        __syncthreads();
    }
    if (!direct) {
        int run = 0;
#pragma unroll
        for (int j = 0; j < kBucketItems; ++j) {
            ++run;
            const int b = c[j] >> g.width_log;  // (-1 stays -1)
            if (j + 1 < kBucketItems && c[j + 1] >> g.width_log == b) continue;
            if (b >= 0) atomicAdd(&s_cnt[b], run);
            run = 0;
        }
    }
    __syncthreads();
    for (int b = tid; b < g.buckets; b += kBucketBlock) g.hist[(int64_t)b * g.tiles + tile] = s_cnt[b];
}

// Every entry to its bucket's place.  A tile is put in order in LDS first, so that a bucket's entries leave as runs (7 of a tile over
// 1172 buckets), which the neighbouring tiles of the XCD complete to lines: stored one by one they were as many requests
// to L2 as entries.  (54 M entries, columns and rows: 472 -> 231 us; columns only 227 -> 113.  Tiles of 16384: 254 and 147, a
// workgroup per CU less; two tiles a workgroup, for half the histogram: 264 and 140.)
template <bool ROWS, bool EDGES>
__global__ __launch_bounds__(kBucketBlock) void bucket_scatter_kernel(const BucketArgs g)
{
    constexpr int NT = kBucketBlock, kPer = kMaxBuckets / NT;
    __shared__ __align__(16) int s_buf[kBucketTile];
    __shared__ int s_start[kMaxBuckets];
    __shared__ int s_delta[kMaxBuckets];  // (and, before it is filled, the scratch of the scans)
    const int64_t n = bucket_entries(g);
    const int64_t tile = xcd_tile(g.tiles), e0 = tile * kBucketTile;
    if (tile < 0 || e0 >= n) return;  // (uniform over the workgroup)
    const int direct = ROWS ? 0 : g.direct[tile];
    const int tid = (int)threadIdx.x, at = tid * kBucketItems;
    int32_t c[kBucketItems], r[ROWS ? kBucketItems : 1];
    load_columns(g, e0 + at, n, c);
    if (direct) return;  // (counted already; asked for together with the entries, so that the others do not wait twice)
    if constexpr (ROWS) {
        tile_rows<NT, kBucketItems>(g.indptr, g.n_rows, g.tile_row, tile, n, s_buf, s_delta);
#pragma unroll
        for (int q = 0; q < kBucketItems / 4; ++q) {
            const int4 v = reinterpret_cast<const int4*>(s_buf + at)[q];
            r[4 * q] = v.x; r[4 * q + 1] = v.y; r[4 * q + 2] = v.z; r[4 * q + 3] = v.w;
        }
    }
    for (int b = tid; b < kMaxBuckets; b += NT) s_start[b] = 0;
    __syncthreads();
    // places within the tile: a run of equal buckets takes its places with one update
    int place[kBucketItems], len[kBucketItems];
#pragma unroll
    for (int j = kBucketItems - 1; j >= 0; --j)
        len[j] = j + 1 < kBucketItems && c[j] >> g.width_log == c[(j + 1) % kBucketItems] >> g.width_log ? len[(j + 1) % kBucketItems] + 1 : 1;
#pragma unroll
    for (int j = 0; j < kBucketItems; ++j) {
        const int b = c[j] >> g.width_log;
        place[j] = 0;
        if (j > 0 && b == c[(j + kBucketItems - 1) % kBucketItems] >> g.width_log) place[j] = place[(j + kBucketItems - 1) % kBucketItems] + 1;
        else if (b >= 0) place[j] = atomicAdd(&s_start[b], len[j]);
    }
    __syncthreads();
    int cnt[kPer], sum = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        cnt[q] = s_start[tid * kPer + q];
        sum += cnt[q];
    }
    int total;
    int run = block_exclusive_scan<NT>(sum, s_delta, &total);
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        s_start[tid * kPer + q] = run;
        if (tid * kPer + q < g.buckets) s_delta[tid * kPer + q] = g.hist[(int64_t)(tid * kPer + q) * g.tiles + tile] - run;
        run += cnt[q];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kBucketItems; ++j) {
        if (c[j] < 0) continue;
        place[j] += s_start[c[j] >> g.width_log];
        s_buf[place[j]] = c[j];
    }
    __syncthreads();
    int to[kBucketItems];
#pragma unroll
    for (int j = 0; j < kBucketItems; ++j) {
        const int i = tid + j * NT;
        to[j] = 0;
        if (i < total) {
            const int col = s_buf[i], b = col >> g.width_log;
            to[j] = i + s_delta[b];
            g.b_col[to[j]] = (uint16_t)(col - (b << g.width_log));
        }
    }
    auto send = [&](int32_t* out, auto value) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kBucketItems; ++j)
            if (c[j] >= 0) s_buf[place[j]] = value(j);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kBucketItems; ++j)
            if (tid + j * NT < total) out[to[j]] = s_buf[tid + j * NT];
    };
    if constexpr (ROWS) send(g.b_row, [&](int j) { return r[j]; });
    if constexpr (EDGES) send(g.b_edge, [&](int j) { return (int)(e0 + at + j); });
}

// One workgroup: the buckets cut into segments of at most g.segment entries.
__global__ __launch_bounds__(1024) void bucket_segments_kernel(const BucketArgs g)
{
    __shared__ int smem[1024 / kWave + 1];
    int carry = 0;
    for (int start = 0; start < g.buckets; start += 1024) {
        const int b = start + (int)threadIdx.x;
        int first = 0, size = 0;
        if (b < g.buckets) {
            first = g.hist[(int64_t)b * g.tiles];
            size = g.hist[(int64_t)(b + 1) * g.tiles] - first;
        }
        const int segs = (size + g.segment - 1) / g.segment;
        int total;
        const int at = carry + block_exclusive_scan<1024>(segs, smem, &total);
        for (int q = 0; q < segs; ++q) {
            int32_t* s = g.segments + 1 + 3 * (at + q);
            s[0] = b;
            s[1] = first + q * g.segment;
            s[2] = size - q * g.segment < g.segment ? size - q * g.segment : g.segment;
        }
        carry += total;
    }
    if (threadIdx.x == 0) g.segments[0] = carry;
}

// a segment's columns counted in LDS and added to the counters; PLACES: the sums before it are its places in the columns
template <bool PLACES>
__global__ __launch_bounds__(kBucketBlock) void bucket_count_kernel(const BucketArgs g)
{
    __shared__ int s_cnt[1 << kMaxWidthLog];
    const int seg = (int)blockIdx.x;
    if (seg >= g.segments[0]) return;
    const int width = 1 << g.width_log;
    const int bucket = g.segments[1 + 3 * seg], first = g.segments[2 + 3 * seg], size = g.segments[3 + 3 * seg];
    const int col0 = bucket << g.width_log;
    for (int c = (int)threadIdx.x; c < width; c += kBucketBlock) s_cnt[c] = 0;
    __syncthreads();
    // eight neighbours a lane, from whole 16-byte pieces of the array (which is padded to them); equal ones counted together
    const int64_t g0 = first / 8, g1 = ((int64_t)first + size + 7) / 8;
    for (int64_t q = g0 + threadIdx.x; q < g1; q += kBucketBlock) {
        const uint4 v = reinterpret_cast<const uint4*>(g.b_col)[q];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        int c[8], run = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int64_t i = q * 8 + j;
            c[j] = i >= first && i < (int64_t)first + size ? (int)((w[j / 2] >> (16 * (j % 2))) & 0xFFFFu) : -1;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            ++run;
            if (j + 1 < 8 && c[(j + 1) % 8] == c[j]) continue;
            if (c[j] >= 0) atomicAdd(&s_cnt[c[j]], run);
            run = 0;
        }
    }
    __syncthreads();
    for (int c = (int)threadIdx.x; c < width; c += kBucketBlock) {
        const int v = s_cnt[c];
        if (v == 0) continue;
        if constexpr (PLACES) g.seg_base[((int64_t)seg << g.width_log) + c] = atomicAdd(&g.counts[(int64_t)col0 + c], v);
        else atomicAdd(&g.counts[(int64_t)col0 + c], v);
    }
}

// ... and, once the counts have become offsets, every entry into its column's row of the transposed block.  A chunk of the segment
// is put in order by column in LDS and leaves as runs: stored one by one, a segment's entries go all over its bucket's 200 KB of
// the output, a thousand segments' worth of which no L2 holds.  (54 M entries: 737 -> 207 us.)
// Entries that are next to each other in the output already -- those of sorted ids, and of a graph whose rows keep to a band -- and segments
// of buckets with fewer entries than columns are stored as they are met: ordering them only lengthens the chain.  (This launch, all segments in order ->
// now, as it was when all were stored: 300 K entries, 6 M columns 55 -> 10, 11; 5 M in a band of 14 M columns 114 -> 35, 31; whole transposes with edge ids, 1.2 M
// sorted entries of 300 K columns 71 -> 61, 60; 30 M of 2.4 M columns, sorted 505 -> 453, 572, in a band 64 wide 480 -> 482, 749, uniform 577 -> 575, 2061.)
constexpr int kLook = 4;    // entries of a lane that a segment is judged by
constexpr int kNear = 200;  // entries of the output that neighbours may lie apart on average: bands 64 wide cross at some ten entries a column
template <int WIDTH_LOG, bool EDGES>
__global__ __launch_bounds__(kBucketBlock) void bucket_fill_kernel(const BucketArgs g)
{
    constexpr int kWidth = 1 << WIDTH_LOG, kPer = kWidth / kBucketBlock;
    __shared__ int s_buf[kBucketTile];
    __shared__ int s_at[kWidth + kBucketBlock];  // by column: entries, their first place in the chunk, what leads from there to the output
    __shared__ int s_scan[kBucketBlock / kWave + 1];
    auto slot = [](int c) { return c + c / kPer; };  // (a lane's columns are neighbours: no two lanes meet in a bank)
    const int seg = (int)blockIdx.x;
    if (seg >= g.segments[0]) return;
    const int bucket = g.segments[1 + 3 * seg], first = g.segments[2 + 3 * seg], size = g.segments[3 + 3 * seg];
    const int tid = (int)threadIdx.x;
    // the segment's next place in each of the lane's columns (columns that it does not mention: never used)
    int next[kPer];
    {
        const int64_t col0 = (int64_t)bucket * kWidth + tid * kPer;
        const int32_t* base = g.seg_base + (int64_t)seg * kWidth + tid * kPer;
        if (col0 + kPer <= g.n_cols) {
            typedef int32_t I4 __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
            for (int q = 0; q < kPer / 4; ++q) {
                const I4 a = reinterpret_cast<const I4*>(g.counts + col0)[q], b = reinterpret_cast<const I4*>(base)[q];
#pragma unroll
                for (int j = 0; j < 4; ++j) next[4 * q + j] = a[j] + b[j];
            }
        } else {
#pragma unroll
            for (int q = 0; q < kPer; ++q) next[q] = col0 + q < g.n_cols ? g.counts[col0 + q] + base[q] : 0;
        }
    }
    // how far apart neighbouring entries' columns lie, from the segment's first entries, and how many entries the bucket's columns have
    const int64_t bucket0 = (int64_t)bucket * kWidth;
    const int64_t entries = (bucket0 + kWidth < g.n_cols ? g.counts[bucket0 + kWidth] : g.n_max) - g.counts[bucket0];
    bool direct = entries < kWidth;
    if (!direct && size >= kLook * kBucketBlock) {  // (uniform over the workgroup)
        int apart = 0;
#pragma unroll
        for (int j = 0; j < kLook; ++j) {
            const int c = g.b_col[(int64_t)first + tid + j * kBucketBlock];
            const int d = c - __shfl_xor(c, 1, kWave);
            apart += d < 0 ? -d : d;
        }
        apart = block_sum_of_lanes<kBucketBlock>(apart, s_scan);
        direct = (int64_t)apart * entries < (int64_t)kNear * kWidth * (kLook * kBucketBlock);
    }
    if (direct) {
#pragma unroll
        for (int q = 0; q < kPer; ++q) s_at[slot(tid * kPer + q)] = next[q];
        __syncthreads();
        constexpr int kInFlight = 4;
        for (int i0 = tid; i0 < size; i0 += kInFlight * kBucketBlock) {
            int c[kInFlight], r[kInFlight], e[kInFlight];
#pragma unroll
            for (int j = 0; j < kInFlight; ++j) {
                const int64_t i = i0 + j * kBucketBlock;
                c[j] = -1;
                if (i < size) {
                    c[j] = g.b_col[first + i];
                    r[j] = g.b_row[first + i];
                    if constexpr (EDGES) e[j] = g.b_edge[first + i];
                }
            }
#pragma unroll
            for (int j = 0; j < kInFlight; ++j) {
                if (c[j] < 0) continue;
                const int at = atomicAdd(&s_at[slot(c[j])], 1);
                g.t_indices[at] = r[j];
                if constexpr (EDGES) g.t_edge[at] = e[j];
            }
        }
        return;
    }
    for (int from = 0; from < size; from += kBucketTile) {
        const int here = size - from < kBucketTile ? size - from : kBucketTile;
        const int64_t e0 = (int64_t)first + from;
        int c[kBucketItems], place[kBucketItems];
#pragma unroll
        for (int j = 0; j < kBucketItems; ++j) {
            const int i = tid + j * kBucketBlock;
            c[j] = i < here ? (int)g.b_col[e0 + i] : -1;
        }
        for (int q = tid; q < kWidth + kBucketBlock; q += kBucketBlock) s_at[q] = 0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kBucketItems; ++j) place[j] = c[j] >= 0 ? atomicAdd(&s_at[slot(c[j])], 1) : 0;
        __syncthreads();
        int cnt[kPer], sum = 0;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            cnt[q] = s_at[slot(tid * kPer + q)];
            sum += cnt[q];
        }
        int total;
        int run = block_exclusive_scan<kBucketBlock>(sum, s_scan, &total);
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            s_at[slot(tid * kPer + q)] = run;
            const int n = cnt[q];
            cnt[q] = next[q] - run;
            next[q] += n;
            run += n;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kBucketItems; ++j) {
            if (c[j] < 0) continue;
            place[j] += s_at[slot(c[j])];
            s_buf[place[j]] = c[j];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kPer; ++q) s_at[slot(tid * kPer + q)] = cnt[q];
        __syncthreads();
        int to[kBucketItems];
#pragma unroll
        for (int j = 0; j < kBucketItems; ++j) {
            const int i = tid + j * kBucketBlock;
            to[j] = i < here ? i + s_at[slot(s_buf[i])] : 0;
        }
        auto send = [&](int32_t* out, const int32_t* in) {  // (one array after the other: registers)
            int v[kBucketItems];
#pragma unroll
            for (int j = 0; j < kBucketItems; ++j) v[j] = tid + j * kBucketBlock < here ? in[e0 + tid + j * kBucketBlock] : 0;
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kBucketItems; ++j)
                if (tid + j * kBucketBlock < here) s_buf[place[j]] = v[j];
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kBucketItems; ++j)
                if (tid + j * kBucketBlock < here) out[to[j]] = s_buf[tid + j * kBucketBlock];
        };
        send(g.t_indices, g.b_row);
        if constexpr (EDGES) send(g.t_edge, g.b_edge);
        __syncthreads();
    }
}

// ---- sizes and launches -----------------------------------------------------------------------------------------
static int range_slices(int64_t n_ids, int64_t n_counters)
{
    const int64_t ranges = ceil_div(n_counters, kRangeCounters);
    int64_t s = 512 / ranges;  // two workgroups per CU
    const int64_t most = ceil_div(n_ids, 16384);
    if (s > most) s = most;
    return (int)(s > 0 ? s : 1);
}

// What the forms measured (us, MI355X, replayed from a graph; atomics / ranges / buckets), counting:
//   75 K ids, 27 K counters, R-MAT          24 /   7 /  -           205 K, 200 K, uniform    11.5 / 14 / 23
//   144 K, 400 K, uniform                    9 /  15 /  -           251 K, 27 K, R-MAT         60 /  9 / 29
//   2.5 M, 100 K, R-MAT                    314 /  24 / 45           3.1 M, 2.4 M, R-MAT       433 /  - / 45
//   54 M, 2.4 M, R-MAT                    5900 /   - / 310          54 M, 2.4 M, sorted     13200 /  - / 270
// Ranges read every id once per range and store every counter once per slice: they are kept to half a million counters (32
// ranges) and four million ids, and small inputs take them where a counter is mentioned twice on average.
static bool count_by_ranges(int64_t n_ids, int64_t n_counters)
{
    return n_ids >= ((int64_t)1 << 16) && n_ids < ((int64_t)1 << 22) && n_counters > 0 && n_counters <= ((int64_t)1 << 19) &&
           (n_ids >= ((int64_t)1 << 18) || 2 * n_counters <= n_ids);
}
static bool fits_buckets(int64_t n_entries, int64_t n_cols) { return n_entries <= 0x7FFFFFFF && n_cols > 0 && n_cols <= ((int64_t)kMaxBuckets << kMaxWidthLog); }
static bool count_by_buckets(int64_t n_ids, int64_t n_counters)
{
    return n_ids >= ((int64_t)1 << 20) && !count_by_ranges(n_ids, n_counters) && fits_buckets(n_ids, n_counters);
}
// Transposing (atomics with the fill by entries / buckets): 205 K entries, 200 K columns, uniform 26 / 43; 251 K, 27 K, R-MAT 88 / 72;
// 434 K, a sampled block 93 / 75; 600 K, 200 K, uniform 47 / 50; 1.15 M, a sampled block 113 / 91; 2.5 M, 100 K, R-MAT 335 / 108;
// 54 M, 2.4 M, R-MAT 24700 (sixteen lanes per row) / 700.  Columns of graphs are skewed: the line is where those gain, and uniform
// ones pay up to twice the time there (300 K entries, 30 K columns 31 / 57, columns drawn as u^4 319 / 67; 600 K, 30 K 47 / 70, 591 / 71;
// 300 K, 300 K 32 / 47, 207 / 70); from 1.2 M on neither does.
bool bucket_transpose_form(int64_t n_entries, int64_t n_cols) { return n_entries >= ((int64_t)1 << 18) && fits_buckets(n_entries, n_cols); }

// Up to two million entries, segments are shorter: those of 32768 are so few that most of the chip waits for them, the longer the more is done for
// each chunk of them.  From 128 buckets on, half as many entries again as a bucket holds on average, so that buckets that are alike are not cut.
// (Transposes with edge ids, us, segments of 32768 / these: 300 K entries, 30 K columns, uniform 69 / 53, in a band 72 / 55; 1.2 M entries, 30 K columns 99 / 70,
// 300 K columns, uniform 66 / 65, drawn as u^3 96 / 73.)
static int segment_entries(int64_t n_entries, int64_t buckets)
{
    if (n_entries > ((int64_t)1 << 21)) return kSegment;
    const int64_t s = buckets < 128 ? kMinSegment : (int64_t)align_up((size_t)(n_entries * 3 / (2 * buckets)), 512);
    return (int)(s < kMinSegment ? kMinSegment : s > kSegment ? kSegment : s);
}

static void bucket_layout(int64_t n_entries, int64_t n_cols, bool rows, bool edges, void* ws, BucketArgs* g, size_t* bytes)
{
    int w = kMinWidthLog;
    while ((n_cols + ((int64_t)1 << w) - 1) >> w > kMaxBuckets) ++w;
    g->width_log = w;
    g->buckets = (int)((n_cols + ((int64_t)1 << w) - 1) >> w);
    g->tiles = ceil_div(n_entries, kBucketTile);
    g->segment = segment_entries(n_entries, g->buckets);
    const int64_t max_segments = g->buckets + n_entries / g->segment + 1;
    Carver c(ws);
    g->hist = c.take<int32_t>((size_t)(g->buckets * g->tiles + 1));
    g->segments = c.take<int32_t>((size_t)(1 + 3 * max_segments));
    g->b_col = c.take<uint16_t>(align_up((size_t)n_entries, 8));  // (read in 16-byte pieces)
    g->direct = rows ? nullptr : c.take<int32_t>((size_t)g->tiles);
    if (rows) {
        g->tile_row = c.take<int32_t>((size_t)g->tiles);
        g->b_row = c.take<int32_t>((size_t)n_entries);
        g->seg_base = c.take<int32_t>((size_t)(max_segments << w));
    }
    if (edges) g->b_edge = c.take<int32_t>((size_t)n_entries);
    *bytes = c.used();
}

size_t bucket_workspace_bytes(int64_t n_entries, int64_t n_cols, bool rows, bool edges)
{
    BucketArgs g;
    size_t bytes;
    bucket_layout(n_entries, n_cols, rows, edges, nullptr, &g, &bytes);
    return bytes;
}

static int launch_partition(const BucketArgs& g, bool rows, bool edges, hipStream_t stream)
{
    int64_t init_items = g.n_cols;
    if (rows && g.n_rows > init_items) init_items = g.n_rows;
    int64_t blocks = ceil_div(init_items, kBlock);
    if (blocks > 8192) blocks = 8192;
    const unsigned tiles = (unsigned)align_up(g.tiles, 8);
    hipLaunchKernelGGL(bucket_init_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, stream, g);
    if (rows) hipLaunchKernelGGL(bucket_hist_kernel<false>, dim3(tiles), dim3(kBucketBlock), 0, stream, g);
    else hipLaunchKernelGGL(bucket_hist_kernel<true>, dim3(tiles), dim3(kBucketBlock), 0, stream, g);
    FGL_CHECK_LAUNCH("bucket_hist_kernel");
    const int64_t n_hist = g.buckets * g.tiles;
    // (the entries are not written yet: the scan's scratch -- a few words per tile -- fits where they go)
    int rc = launch_exclusive_sum(g.hist, n_hist, nullptr, g.hist, nullptr, g.b_col, scan_workspace_bytes(n_hist), stream);
    if (rc != FGL_OK) return rc;
    if (rows && edges) hipLaunchKernelGGL((bucket_scatter_kernel<true, true>), dim3(tiles), dim3(kBucketBlock), 0, stream, g);
    else if (rows) hipLaunchKernelGGL((bucket_scatter_kernel<true, false>), dim3(tiles), dim3(kBucketBlock), 0, stream, g);
    else hipLaunchKernelGGL((bucket_scatter_kernel<false, false>), dim3(tiles), dim3(kBucketBlock), 0, stream, g);
    hipLaunchKernelGGL(bucket_segments_kernel, dim3(1), dim3(1024), 0, stream, g);
    const unsigned segs = (unsigned)(g.buckets + g.n_max / g.segment + 1);
    if (rows) hipLaunchKernelGGL(bucket_count_kernel<true>, dim3(segs), dim3(kBucketBlock), 0, stream, g);
    else hipLaunchKernelGGL(bucket_count_kernel<false>, dim3(segs), dim3(kBucketBlock), 0, stream, g);
    FGL_CHECK_LAUNCH("bucket_count_kernel");
    return FGL_OK;
}

size_t count_workspace_bytes(int64_t n_ids, int64_t n_counters)
{
    if (count_by_buckets(n_ids, n_counters)) return bucket_workspace_bytes(n_ids, n_counters, false, false);
    if (count_by_ranges(n_ids, n_counters)) return align_up((size_t)range_slices(n_ids, n_counters) * n_counters * sizeof(int32_t), 256);
    return 0;
}

// counts[0 .. n_counters) of the ids; false if this size has no form here (the caller counts with atomics)
bool launch_count(const int32_t* d_ids, int64_t n_ids, const int32_t* d_n, int64_t n_counters, int32_t* d_counts, void* d_ws,
                  hipStream_t stream, int* rc)
{
    *rc = FGL_OK;
    if (count_by_buckets(n_ids, n_counters)) {
        BucketArgs g;
        memset(&g, 0, sizeof(g));
        size_t bytes;
        bucket_layout(n_ids, n_counters, false, false, d_ws, &g, &bytes);
        g.ids = d_ids; g.n_max = n_ids; g.d_n = d_n; g.n_cols = n_counters; g.counts = d_counts;
        *rc = launch_partition(g, false, false, stream);
        return true;
    }
    if (!count_by_ranges(n_ids, n_counters)) return false;
    const int slices = range_slices(n_ids, n_counters);
    int32_t* partial = static_cast<int32_t*>(d_ws);
    hipLaunchKernelGGL(count_ranges_kernel, dim3((unsigned)ceil_div(n_counters, kRangeCounters), (unsigned)slices), dim3(kRangeBlock), 0, stream,
                       d_ids, n_ids, d_n, ceil_div(n_ids, slices), n_counters, partial);
    hipLaunchKernelGGL(count_ranges_sum_kernel, dim3((unsigned)ceil_div(n_counters, kBlock)), dim3(kBlock), 0, stream, partial, slices,
                       n_counters, d_counts);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("count_ranges_kernel: launch failed: %s", hipGetErrorString(e));
        *rc = FGL_ERR_HIP;
    }
    return true;
}

// d_t_indptr, d_t_indices and d_t_edge (may be null) of the transposed block; *d_longest (may be null) becomes zero.
int launch_bucket_transpose(const int32_t* d_indptr, const int32_t* d_indices, int64_t n_rows, int64_t n_cols, int64_t n_edges,
                            int32_t* d_t_indptr, int32_t* d_t_indices, int32_t* d_t_edge, int32_t* d_longest, void* d_ws, hipStream_t stream)
{
    BucketArgs g;
    memset(&g, 0, sizeof(g));
    size_t bytes;
    const bool edges = d_t_edge != nullptr;
    bucket_layout(n_edges, n_cols, true, edges, d_ws, &g, &bytes);
    g.ids = d_indices; g.n_max = n_edges; g.indptr = d_indptr; g.n_rows = n_rows; g.n_cols = n_cols;
    g.counts = d_t_indptr; g.longest = d_longest; g.t_indices = d_t_indices; g.t_edge = d_t_edge;
    int rc = launch_partition(g, true, edges, stream);
    if (rc != FGL_OK) return rc;
    // (the histogram is no longer needed: scratch of this scan)
    rc = launch_exclusive_sum(d_t_indptr, n_cols, nullptr, d_t_indptr, nullptr, g.hist, scan_workspace_bytes(n_cols), stream);
    if (rc != FGL_OK) return rc;
    const unsigned segs = (unsigned)(g.buckets + n_edges / g.segment + 1);
#define FGL_LAUNCH_FILL(W)                                                                                                   \
    do {                                                                                                                      \
        if (edges) hipLaunchKernelGGL((bucket_fill_kernel<W, true>), dim3(segs), dim3(kBucketBlock), 0, stream, g);             \
        else hipLaunchKernelGGL((bucket_fill_kernel<W, false>), dim3(segs), dim3(kBucketBlock), 0, stream, g);                  \
    } while (0)
    static_assert(kMaxWidthLog == kMinWidthLog + 2, "a form of the kernel for each width");
    if (g.width_log == kMinWidthLog) FGL_LAUNCH_FILL(kMinWidthLog);
    else if (g.width_log == kMinWidthLog + 1) FGL_LAUNCH_FILL(kMinWidthLog + 1);
    else FGL_LAUNCH_FILL(kMaxWidthLog);
#undef FGL_LAUNCH_FILL
    FGL_CHECK_LAUNCH("bucket_fill_kernel");
    return FGL_OK;
}

}  // namespace fgl
