// Fused id-map: open-addressing hash table over global node ids (stands in for the
// reference's Entry table and its four kernels, cuda_operators/id_map.cu:26-59,179-383).
//
// Slot = 8 bytes {uint32 key, uint32 val}, empty = all ones.  Slot count is a power of two,
// hash = (id * 0x9E3779B1) >> (32 - log2 slots), linear probing (8 slots per 64-byte line),
// every probe loop bounded by the slot count.  `val` is the node's local id once the id is
// numbered; while a batch of new ids is being numbered it transiently holds
// kPending | (index of the first edge that mentions the id), maintained with atomicMin, so that
// new ids are numbered in first-occurrence order -- deterministic, and the order DGL's
// to_block gives -- instead of the reference's race on one global counter (id_map.cu:317-320).
//
// map_src = two launches (three beyond 1 M edges, four beyond 8 M):
//   1. insert     per edge: probe (one 8-byte load per slot), install {key, pending first-edge index}
//                 with one 64-bit CAS if new, else atomicMin the first-edge index; remember the slot.
//                 An id that was numbered before this call is relabelled on the spot from the val
//                 the probe has loaded anyway, and the edge takes no further part.
//                 The edges that are first mentions of new ids are kept track of as they change, a bit
//                 per edge (MentionMarks, mark_first).  In a mini-batch's small hops the sampling kernel
//                 does this itself with the edges it has just drawn.
//   2. number     per edge: an edge whose bit is set is its id's first mention, and its local id is the
//                 number of bits before it: a prefix per 512 edges (64 bytes of bits, which every
//                 workgroup counts and scans into LDS for itself) plus the bits of its own line.  It appends
//                 the id to the unique list and stores the local id in the id's slot for later calls --
//                 skipped with FGL_IDMAP_FINAL, when the caller will not consult the table again (the last
//                 hop of a mini-batch: most of its edges).  Any other edge reads its slot: the local id, if
//                 the first mention's lane has been there already, else the index of that first mention,
//                 and counts the bits before that.
//   (count)       larger inputs: the bits counted once, per line and per 4096 edges; the number pass then scans
//                 the latter only
//   (prefix)      ... and where even those are too many for every workgroup, a single workgroup scans them
#include "fgl_common.hpp"
#include "fgl_kernels.hpp"
#include "fgl_table.hpp"
#include "fgl_transpose_job.hpp"
#include "fgl_idmap_device.hpp"

namespace fgl {

__global__ __launch_bounds__(kBlock) void idmap_insert_dst_kernel(TableRef t, const int32_t* __restrict__ ids,
                                                                  int64_t n_max, const int32_t* __restrict__ d_n,
                                                                  int32_t* __restrict__ uniq, uint32_t* __restrict__ d_status,
                                                                  uint32_t* __restrict__ zero_words, int64_t n_zero_words)
{
    const int64_t n = actual_count(n_max, d_n);
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    // (scratch of the passes that follow in the same call, cleared on the way)
    for (int64_t w = i; w < n_zero_words; w += (int64_t)gridDim.x * kBlock) zero_words[w] = 0u;
    if (i >= n) return;
    const int32_t id = ids[i];
    if (uniq != nullptr && uniq != ids) uniq[i] = id;
    if (id < 0) {  // not a node id (and -1 would read as the empty marker): reported, never inserted
        if (d_status) atomicOr(d_status, FGL_STATUS_BAD_ID);
        return;
    }
    uint32_t seen;
    const uint32_t p = find_or_insert(t, (uint32_t)id, (uint32_t)i, &seen);  // a repeated id keeps its first position
    if (p == kEmpty && d_status) atomicOr(d_status, FGL_STATUS_TABLE_FULL);
}

// One edge per lane: the pass is bound by the rate at which the chip retires atomics, and several edges in flight per lane only
// take parallelism away (a hop of 1.5 M edges on a 111 M-node graph: 1 edge 56 us, 2 -> 62 us, 4 -> 70 us).
// `src` and `out` may be the same array (relabelling in place): neither is __restrict__.
__global__ __launch_bounds__(kBlock) void idmap_insert_src_kernel(const int32_t* src, int64_t e_max, const int32_t* __restrict__ d_e,
                                                                  const InsertWork w, uint32_t* __restrict__ d_status, int32_t* dst_inout)
{
    unsigned long long* slots = reinterpret_cast<unsigned long long*>(w.t.words);
    const int64_t n_e = actual_count(e_max, d_e);
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t base = (int64_t)blockIdx.x * kBlock; base < n_e; base += stride) {
        const int64_t e = base + threadIdx.x;
        const int32_t id = e < n_e ? src[e] : -1;
        const uint32_t p = ((uint32_t)id * kHashMul) >> w.t.shift;
        const unsigned long long s = id >= 0 ? slots[p] : 0ull;
        // The destination half of transfer_edge_id (id_map.cu:377-381) rides on this pass when the caller asks: the
        // edge's destination id -- numbered by an earlier launch -- is looked up and relabelled in place, its first
        // probe travelling together with the source id's.
        if (dst_inout != nullptr && e < n_e) {
            const uint32_t d = (uint32_t)dst_inout[e];
            int32_t local = -1;
            if ((int32_t)d >= 0) {
                uint32_t q = (d * kHashMul) >> w.t.shift;
                const uint32_t limit = w.t.mask < kMaxProbes ? w.t.mask + 1 : kMaxProbes;
                for (uint32_t n = 0; n < limit; ++n) {
                    const unsigned long long v = slots[q];
                    if ((uint32_t)v == d) {
                        // (a destination id holds its number; one that only an edge of this call has mentioned
                        // so far -- pending -- is not a destination: missing)
                        if (!((uint32_t)(v >> 32) & kPending)) local = (int32_t)(v >> 32);
                        break;
                    }
                    if ((uint32_t)v == kEmpty) break;
                    q = (q + 1) & w.t.mask;
                }
            }
            if (local < 0 && d_status) atomicOr(d_status, FGL_STATUS_MISSING_KEY);
            dst_inout[e] = local;
        }
        bool holder = false;
        if (e < n_e) {
            uint32_t seen = 0, displaced = kEmpty, q = kEmpty;
            if (id >= 0) q = insert_mention_from(w.t, (uint32_t)id, kPending | (uint32_t)e, p, s, &seen, &holder, &displaced);
            finish_insert(w, e, n_e, id, q, seen, displaced, d_status);
        }
        mark_first(w.marks, base + threadIdx.x / kWave * kWave, holder);
    }
}

// n_total = n_base + (number of new ids), clamped to the capacity of the unique list.
// readback (optional, may be host memory that the device can write): where the host reads the call's sizes.
// Without rb_counts: two words, {node total, status word}.  With rb_counts (the all-hops call's count array, which
// holds both d_n_total_out and the status word): a copy of its rb_n words as they stand now -- the other entries
// were final before this launch began.
__device__ __forceinline__ void publish_node_total(int64_t n_base, int n_new, int64_t capacity,
                                                   int32_t* __restrict__ d_n_total_out, uint32_t* __restrict__ d_status,
                                                   int32_t* __restrict__ readback = nullptr,
                                                   const int32_t* __restrict__ rb_counts = nullptr, int rb_n = 0)
{
    int64_t total = n_base + (int64_t)n_new;
    uint32_t overflow = 0u;
    if (total > capacity) {
        overflow = FGL_STATUS_UNIQ_OVERFLOW;
        if (d_status) atomicOr(d_status, FGL_STATUS_UNIQ_OVERFLOW);
        total = capacity;
    }
    if (d_n_total_out) *d_n_total_out = (int32_t)total;
    if (readback == nullptr) return;
    // (every other bit of the status word was set by an earlier launch of the call)
    const int32_t status = (int32_t)((d_status ? *d_status : 0u) | overflow);
    if (rb_counts == nullptr) {
        readback[0] = (int32_t)total;
        readback[1] = status;
        return;
    }
    for (int i = 0; i < rb_n; ++i) {
        int32_t v = rb_counts[i];
        if (rb_counts + i == d_n_total_out) v = (int32_t)total;
        if (rb_counts + i == reinterpret_cast<const int32_t*>(d_status)) v = status;
        readback[i] = v;
    }
}

// One workgroup: exclusive scan of the per-tile counts of new ids, then
// n_total = n_base + (number of new ids), clamped to the capacity of the unique list.
__global__ __launch_bounds__(1024) void idmap_prefix_publish_kernel(const int32_t* __restrict__ tile_sums,
                                                                    int32_t* __restrict__ tile_prefix, int64_t e_max,
                                                                    const int32_t* __restrict__ d_e, int64_t n_base_h,
                                                                    const int32_t* __restrict__ d_n_base, int64_t capacity,
                                                                    int32_t* __restrict__ d_n_total_out,
                                                                    uint32_t* __restrict__ d_status, int32_t* __restrict__ readback,
                                                                    const int32_t* __restrict__ rb_counts, int rb_n)
{
    __shared__ int smem[1024 / kWave + 1];
    const int n_tiles = (int)mark_tiles(actual_count(e_max, d_e));
    int carry = 0;
    for (int start = 0; start < n_tiles; start += 1024) {
        const int i = start + (int)threadIdx.x;
        const int v = i < n_tiles ? tile_sums[i] : 0;
        int total;
        const int ex = block_exclusive_scan<1024>(v, smem, &total);
        if (i < n_tiles) tile_prefix[i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0)
        publish_node_total(d_n_base ? (int64_t)(*d_n_base) : n_base_h, carry, capacity, d_n_total_out, d_status, readback, rb_counts, rb_n);
}

// How a number pass comes by the marks before a line of edges (kMode):
//   kFromBits     every workgroup counts all lines' bits itself and scans the counts in LDS: up to kLinesInLds lines, i.e. one
//                 launch fewer where launches, not edges, set the time (128 KB of bits a workgroup at most);
//   kFromTiles    a count launch has counted lines and tiles of eight lines; every workgroup scans the tiles' counts in LDS;
//   kFromPrefix   as kFromTiles, with a prefix launch behind the count launch that has scanned them.
// In the first two the first workgroup publishes the node total.
constexpr int kFromBits = 0, kFromTiles = 1, kFromPrefix = 2;
constexpr int kEntriesPerLane = 8;
constexpr int kLinesInLds = kBlock * kEntriesPerLane;
constexpr int kNumberMaxBlocks = 1024;

// eight lanes per tile of 4096 edges, a line each
__global__ __launch_bounds__(kBlock) void idmap_count_kernel(const MentionMarks marks, int64_t e_max, const int32_t* __restrict__ d_e,
                                                             int32_t* __restrict__ line_counts, int32_t* __restrict__ tile_sums)
{
    const int64_t n_lines = mark_tiles(actual_count(e_max, d_e)) * (kMarkTile / kMarkLine);
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t line = (int64_t)blockIdx.x * kBlock + threadIdx.x; line < n_lines; line += stride) {  // (eight lanes at a time)
        int c = line_count(marks, line);
        line_counts[line] = c;
#pragma unroll
        for (int d = 1; d < kMarkTile / kMarkLine; d <<= 1) c += __shfl_xor(c, d, kWave);
        if (line % (kMarkTile / kMarkLine) == 0) tile_sums[line / (kMarkTile / kMarkLine)] = c;
    }
}

// The new nodes that the lanes of a wave number in one step have consecutive positions (a position is a count of
// earlier new nodes, and the lanes hold consecutive edges), so their tiles of the next hop are at most two:
// one atomic per tile and wave instead of one per node -- updates of one address run one after the other, and a
// tile's 256 nodes would otherwise queue up on it.  k = 0 for lanes without a new node.  Every lane of the wave
// must call this.
__device__ __forceinline__ void add_next_tile_sums(const NextHop& next, int k, int tile)
{
    if (__ballot(k != 0) == 0) return;  // uniform
    int tmin = k != 0 ? tile : 0x7FFFFFFF;
#pragma unroll
    for (int d = kWave / 2; d >= 1; d >>= 1) {
        const int o = __shfl_xor(tmin, d, kWave);
        tmin = o < tmin ? o : tmin;
    }
    int s0 = (k != 0 && tile == tmin) ? k : 0;
    int s1 = (k != 0 && tile != tmin) ? k : 0;
#pragma unroll
    for (int d = kWave / 2; d >= 1; d >>= 1) {
        s0 += __shfl_xor(s0, d, kWave);
        s1 += __shfl_xor(s1, d, kWave);
    }
    if (lane_id() == 0) {
        atomicAdd(&next.tile_sums[tmin], s0);
        if (s1 != 0) atomicAdd(&next.tile_sums[tmin + 1], s1);
    }
}

// Lane per edge, coalesced.  `src` and `out` may be the same array: an entry is read and written by one lane only.
// (Edges whose id was numbered before this call were relabelled by the insert pass.)  A first mention's local id is the number
// of marks before its edge; it appends the id to the unique list and, unless the caller has said that the table will not be
// consulted again (WRITE_BACK = false), stores the local id in the id's slot.  The other edges of new ids -- a fifth to two
// fifths of a hop's -- read the slot: it holds the local id already, or still the index of the first mention.
// (A pass between insert and number used to read every edge's slot, flag the first mentions and count them: 5.3-6.6 us of a small
// hop's three launches, 10.4 us for 1.5 M edges; this pass took 17.7 us for those, now 19.2 + 4.7 for the count.)
// The launch also carries (in workgroups behind its own) what the hops around it need: `scan` turns the counters of the hop
// before's transposed block into offsets, `zero` and zero_marks clear the counters and marks of the next hop.
template <int kMode, bool WRITE_BACK>
__global__ __launch_bounds__(kBlock) void idmap_number_kernel(TableRef t, const int32_t* src, int64_t e_max,
                                                              const int32_t* __restrict__ d_e, int64_t n_base_h,
                                                              const int32_t* __restrict__ d_n_base,
                                                              const uint32_t* __restrict__ slot_of, const MentionMarks marks,
                                                              const int32_t* __restrict__ line_counts,
                                                              const int32_t* __restrict__ tile_counts,  // kFromPrefix: their prefixes
                                                              int32_t* __restrict__ uniq, int64_t capacity, int32_t* out,
                                                              int32_t* __restrict__ d_n_total_out,
                                                              uint32_t* __restrict__ d_status, const NextHop next,
                                                              const TransposeRank tr, const TransposeJob scan, const TransposeJob zero,
                                                              const ZeroJob zero_marks, int n_side, int32_t* __restrict__ readback,
                                                              const int32_t* __restrict__ rb_counts, int rb_n)
{
    __shared__ int s_prefix[kMode != kFromPrefix ? kLinesInLds : 1];
    __shared__ int smem[kBlock / kWave + 1];
    tjob_scan<kBlock>(scan);
    tjob_zero<kBlock>(zero);
    zero_job<kBlock>(zero_marks);
    const int64_t own_blocks = (int64_t)gridDim.x - n_side;
    if ((int64_t)blockIdx.x >= own_blocks) return;
    const int64_t n_e = actual_count(e_max, d_e);
    const int64_t n_base = d_n_base ? (int64_t)(*d_n_base) : n_base_h;
    const int64_t stride = own_blocks * kBlock;
    if ((int64_t)blockIdx.x * kBlock >= n_e && blockIdx.x != 0) return;  // (workgroup 0 publishes the total in any case)
    // What the first trip of the loop below reads about its edge is fetched now, so that it travels together with
    // the counts that the scan waits for (a small hop is one trip per workgroup: a chain of memory latencies).
    uint32_t p_ahead = kDone;
    unsigned long long bits_ahead = 0;
    int32_t id_ahead = 0;
    {
        const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
        if (e < n_e) {
            p_ahead = slot_of[e];
            bits_ahead = marks.bits[e >> 6];
            id_ahead = src[e];
        }
    }
    if constexpr (kMode != kFromPrefix) {
        // (<= kLinesInLds entries: the launcher checks the bound)
        const int n_entries = (int)(kMode == kFromBits ? (n_e + kMarkLine - 1) / kMarkLine : mark_tiles(n_e));
        const int n_used = (n_entries + kBlock - 1) / kBlock * kBlock;
        for (int i = threadIdx.x; i < n_used; i += kBlock)
            s_prefix[i] = i < n_entries ? (kMode == kFromBits ? line_count(marks, i) : tile_counts[i]) : 0;
        __syncthreads();
        const int per_lane = n_used / kBlock;  // <= kEntriesPerLane
        int s = 0;
        for (int j = 0; j < per_lane; ++j) s += s_prefix[(int)threadIdx.x * per_lane + j];
        int total;
        int run = block_exclusive_scan<kBlock>(s, smem, &total);
        for (int j = 0; j < per_lane; ++j) {
            const int c = s_prefix[(int)threadIdx.x * per_lane + j];
            s_prefix[(int)threadIdx.x * per_lane + j] = run;
            run += c;
        }
        __syncthreads();
        if (blockIdx.x == 0 && threadIdx.x == 0) publish_node_total(n_base, total, capacity, d_n_total_out, d_status, readback, rb_counts, rb_n);
    }
    // (the trip count is the same for all lanes of a wave: they add up their next-hop tile sums together)
    for (int64_t base = (int64_t)blockIdx.x * kBlock; base < n_e; base += stride) {
        const int64_t e = base + threadIdx.x;
        int next_k = 0, next_tile = 0;
        const bool first_trip = base == (int64_t)blockIdx.x * kBlock;
        const uint32_t p = first_trip ? p_ahead : (e < n_e ? slot_of[e] : kDone);
        const unsigned long long bits = first_trip ? bits_ahead : (e < n_e ? marks.bits[e >> 6] : 0ull);
        const bool is_first = p < kDone && ((bits >> (e & 63)) & 1ull);
        int32_t id = 0;
        if (is_first) id = first_trip ? id_ahead : src[e];
        int64_t row_a = kRowBadId, row_deg = 0;
        if (next.row_start != nullptr && is_first) load_row_of(next, id, &row_a, &row_deg);
        if (p != kDone) {
            int64_t local = -1;
            if (p < kDone) {
                int64_t ef = e;
                if (!is_first) {
                    const uint32_t v = t.words[2 * (size_t)p + 1];
                    if (v & kPending) ef = (int64_t)(v & ~kPending);  // first edge of this edge's id (< e)
                    else {
                        local = v;
                        ef = n_e;
                    }
                }
                if (ef < n_e) {
                    local = n_base + marks_before_in_line(marks, ef);
                    if (kMode == kFromBits) {
                        local += s_prefix[ef / kMarkLine];
                    } else {
                        const int64_t tile = ef / kMarkTile;
                        local += kMode == kFromTiles ? s_prefix[tile] : tile_counts[tile];
                        const int4* c = reinterpret_cast<const int4*>(line_counts + tile * (kMarkTile / kMarkLine));
                        const int4 a = c[0], b = c[1];
                        const int before[7] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z};
#pragma unroll
                        for (int j = 0; j < 7; ++j) local += j < (int)(ef / kMarkLine % (kMarkTile / kMarkLine)) ? before[j] : 0;
                    }
                }
                if (local < 0 || local >= capacity) local = -1;  // the unique list is full (reported with the node total)
                if (is_first && local < 0) {
                    // (left unnumbered, and without an edge's index: a later hop that meets the id must not take this hop's
                    // edge for one of its own)
                    if (WRITE_BACK) t.words[2 * (size_t)p + 1] = kEmpty;
                } else if (is_first) {
                    uniq[local] = id;
                    if (WRITE_BACK) t.words[2 * (size_t)p + 1] = (uint32_t)local;
                    if (next.row_start != nullptr) {
                        next_k = store_next_hop(next, local, row_a, row_deg);
                        next_tile = (int)(local / next.tile_seeds);
                    }
                }
            }
            out[e] = (int32_t)local;
            take_rank(tr, e, (int32_t)local);
        }
        if (next.row_start != nullptr) add_next_tile_sums(next, next_k, next_tile);
    }
}

__global__ __launch_bounds__(kBlock) void idmap_lookup_kernel(TableRef t, int32_t* __restrict__ ids, int64_t n_max,
                                                              const int32_t* __restrict__ d_n, uint32_t* __restrict__ d_status)
{
    const int64_t n = actual_count(n_max, d_n);
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        const uint32_t p = find_only(t.words, t.mask, t.shift, (uint32_t)ids[i]);
        if (p == kEmpty) {
            if (d_status) atomicOr(d_status, FGL_STATUS_MISSING_KEY);
            ids[i] = -1;
        } else {
            ids[i] = (int32_t)t.words[2 * (size_t)p + 1];
        }
    }
}

// ---- arrival-order numbering (FGL_IDMAP_ARRIVAL) ---------------------------------------
// The lane whose CAS installs a key numbers it at once from a global counter, as the
// reference does (id_map.cu:314-321) -- but with one counter update per workgroup instead
// of one per new id -- and relabels its edge on the spot; so does every lane that finds its id
// already numbered (a destination, an id of an earlier hop, or a new id whose number has landed).
// Only the lanes that meet a key between its install and its number (val still all ones) leave
// their edge to the second, short pass.  Two passes over the edges, one table access per edge in
// most cases; the numbering of new ids depends on scheduling (any run is a valid map, and equal
// to every other after sorting the new ids).  `src` and `out` may be the same array.
template <int ITEMS>
__global__ __launch_bounds__(kBlock) void idmap_insert_arrival_kernel(TableRef t, const int32_t* src,
                                                                      int64_t e_max, const int32_t* __restrict__ d_e,
                                                                      int64_t n_base_h, const int32_t* __restrict__ d_n_base,
                                                                      uint32_t* __restrict__ slot_of, int32_t* __restrict__ counter,
                                                                      int32_t* __restrict__ uniq, int64_t capacity, int32_t* out,
                                                                      uint32_t* __restrict__ d_status, const NextHop next,
                                                                      const TransposeRank tr)
{
    __shared__ int smem[kBlock / kWave + 1];
    __shared__ int s_base;
    constexpr int kNextTiles = kBlock * ITEMS / kWave + 2;  // next-hop tiles (64 seeds or more each) that a tile's new nodes can touch
    __shared__ int s_next[kNextTiles];
    unsigned long long* slots = reinterpret_cast<unsigned long long*>(t.words);
    const int64_t n_e = actual_count(e_max, d_e);
    const int64_t n_base = d_n_base ? (int64_t)(*d_n_base) : n_base_h;
    constexpr int kEdges = kBlock * ITEMS;
    const int64_t n_tiles = (n_e + kEdges - 1) / kEdges;
    const uint32_t limit = t.mask < kMaxProbes ? t.mask + 1 : kMaxProbes;
    // A workgroup takes a tile of 256 * ITEMS edges at a time, ITEMS per lane (edge = tile start + j * 256 + lane).
    // Several edges per lane for large inputs: one update of the global counter per tile -- updates of one address
    // run one after the other, and one per 256 edges costs more than the probing -- against the length of a
    // lane's chain of probes; one edge per lane for small inputs, which need the workgroups.
    // (The trip count is the same for every lane of the workgroup: the loop holds barriers.)
    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int64_t first = tile * kEdges + threadIdx.x;
        // p: kDone = the edge is relabelled; a slot = its id is being numbered, see the second pass; kEmpty = table full
        uint32_t p[ITEMS], id[ITEMS];
        uint32_t won = 0;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int64_t e = first + (int64_t)j * kBlock;
            p[j] = kDone;
            id[j] = 0;
            if (e < n_e) {
                id[j] = (uint32_t)src[e];
                p[j] = kEmpty;
                uint32_t q = (id[j] * kHashMul) >> t.shift;
                // (a negative id is not a node id -- and -1 would read as the empty marker: no probe, reported below)
                for (uint32_t n = 0; n < ((int32_t)id[j] >= 0 ? limit : 0u); ++n) {
                    unsigned long long slot = slots[q];
                    if ((uint32_t)slot == kEmpty) {
                        // the key goes in with val still all ones = "not numbered yet"
                        const unsigned long long seen = atomicCAS(&slots[q], ~0ull, (unsigned long long)id[j] | 0xFFFFFFFF00000000ull);
                        if (seen == ~0ull) {
                            won |= 1u << j;
                            p[j] = q;
                            break;
                        }
                        slot = seen;
                    }
                    if ((uint32_t)slot == id[j]) {
                        const uint32_t v = (uint32_t)(slot >> 32);
                        if (v & 0x80000000u) {
                            p[j] = q;
                        } else {
                            out[e] = (int32_t)v;
                            take_rank(tr, e, (int32_t)v);
                            p[j] = kDone;
                        }
                        break;
                    }
                    q = (q + 1) & t.mask;
                }
                if (p[j] == kEmpty) {
                    out[e] = -1;
                    take_rank(tr, e, -1);
                    if (d_status) atomicOr(d_status, (int32_t)id[j] >= 0 ? FGL_STATUS_TABLE_FULL : FGL_STATUS_BAD_ID);
                }
            }
        }
        // the new nodes' rows in the graph (for the next hop) are fetched while the workgroup takes its numbers
        int64_t row_a[ITEMS], row_deg[ITEMS];
        if (next.row_start != nullptr) {
#pragma unroll
            for (int j = 0; j < ITEMS; ++j)
                if ((won >> j) & 1u) load_row_of(next, (int32_t)id[j], &row_a[j], &row_deg[j]);
        }
        int total;
        int rank = block_exclusive_scan<kBlock>(__popc(won), smem, &total);
        if (threadIdx.x == 0) s_base = total ? atomicAdd(counter, total) : 0;
        if (next.row_start != nullptr)
            for (int i = threadIdx.x; i < kNextTiles; i += kBlock) s_next[i] = 0;
        __syncthreads();
        const int64_t base = n_base + s_base;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int64_t e = first + (int64_t)j * kBlock;
            if ((won >> j) & 1u) {
                const int64_t local = base + rank++;
                if (local < capacity) {
                    t.words[2 * (size_t)p[j] + 1] = (uint32_t)local;
                    uniq[local] = (int32_t)id[j];
                    out[e] = (int32_t)local;
                    take_rank(tr, e, (int32_t)local);
                    if (next.row_start != nullptr) {
                        // (the tile's new nodes have consecutive positions: few next-hop tiles, summed in LDS first)
                        const int k = store_next_hop(next, local, row_a[j], row_deg[j]);
                        if (k != 0) atomicAdd(&s_next[(int)(local / next.tile_seeds - base / next.tile_seeds)], k);
                    }
                } else {
                    out[e] = -1;  // the unique list is full (reported by the second pass); val stays "not numbered"
                    take_rank(tr, e, -1);
                }
                p[j] = kDone;
            }
            if (e < n_e) slot_of[e] = p[j];
        }
        __syncthreads();
        if (next.row_start != nullptr) {
            for (int i = threadIdx.x; i < kNextTiles; i += kBlock)
                if (s_next[i] != 0) atomicAdd(&next.tile_sums[base / next.tile_seeds + i], s_next[i]);
            __syncthreads();  // s_next is cleared again at the top of the next tile
        }
    }
}

// Second pass of the arrival-order numbering: the edges whose id was between install and number when
// their lane met it read the number now; also publishes the node total.
__global__ __launch_bounds__(kBlock) void idmap_relabel_publish_kernel(TableRef t, int64_t e_max, const int32_t* __restrict__ d_e,
                                                                       const uint32_t* __restrict__ slot_of,
                                                                       int32_t* __restrict__ out, const int32_t* __restrict__ counter,
                                                                       int64_t n_base_h, const int32_t* __restrict__ d_n_base,
                                                                       int64_t capacity, int32_t* __restrict__ d_n_total_out,
                                                                       uint32_t* __restrict__ d_status, const TransposeRank tr,
                                                                       const TransposeJob scan, const TransposeJob zero,
                                                                       int32_t* __restrict__ readback,
                                                                       const int32_t* __restrict__ rb_counts, int rb_n)
{
    tjob_scan<kBlock>(scan);  // (carried along for the hops around this one, as in idmap_number_kernel)
    tjob_zero<kBlock>(zero);
    const int64_t n_e = actual_count(e_max, d_e);
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < n_e; e += stride) {
        const uint32_t p = slot_of[e];
        if (p >= kDone) continue;  // relabelled by the first pass (kDone) or reported there (kEmpty)
        const uint32_t v = t.words[2 * (size_t)p + 1];
        const int32_t local = (v & 0x80000000u) ? -1 : (int32_t)v;  // (still unnumbered: the unique list was full)
        out[e] = local;
        take_rank(tr, e, local);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const int64_t n_base = d_n_base ? (int64_t)(*d_n_base) : n_base_h;
        publish_node_total(n_base, *counter, capacity, d_n_total_out, d_status, readback, rb_counts, rb_n);
    }
}

// Inputs up to this many edges number their new ids one edge per lane (see idmap_insert_arrival_kernel).
constexpr int64_t kArrivalSmallEdges = 1 << 18;
constexpr int kArrivalItems = 4;  // edges per lane for large inputs (measured on a 1.5 M-edge hop: 8 -> 69 us, 4 -> 62 us, 2 -> 66 us, 1 -> 100 us)

// Workgroups for a grid-stride pass over n items: enough to fill every CU several times
// over, never more than the work needs.
static inline unsigned stride_grid(int64_t n_items, int items_per_block)
{
    int64_t blocks = ceil_div(n_items > 0 ? n_items : 1, items_per_block);
    if (blocks > 8192) blocks = 8192;
    return (unsigned)blocks;
}

// ---- launchers ------------------------------------------------------------------
int launch_idmap_reset(void* d_table, int64_t slots, hipStream_t stream)
{
    FGL_REQUIRE(d_table != nullptr && valid_slots(slots), "idmap: slot count %lld is not a power of two in [64, 2^31]", (long long)slots);
    return launch_fill_u32(static_cast<uint32_t*>(d_table), slots * 2, kEmpty, stream);
}

int launch_idmap_insert_dst(void* d_table, int64_t slots, const int32_t* d_dst_ids, int64_t n_max, const int32_t* d_n,
                            int32_t* d_uniq, uint32_t* d_status, hipStream_t stream, uint32_t* d_zero_words, int64_t n_zero_words)
{
    FGL_REQUIRE(d_table != nullptr && valid_slots(slots), "idmap: slot count %lld is not a power of two in [64, 2^31]", (long long)slots);
    FGL_REQUIRE(n_max >= 0 && n_max <= slots / 2, "idmap_insert_dst: %lld ids do not fit %lld slots at load 1/2", (long long)n_max, (long long)slots);
    FGL_REQUIRE(n_max <= 0x7FFFFFFF, "idmap_insert_dst: too many ids");
    if (d_zero_words == nullptr) n_zero_words = 0;
    if (n_max == 0 && n_zero_words == 0) return FGL_OK;
    FGL_REQUIRE(n_max == 0 || d_dst_ids != nullptr, "idmap_insert_dst: null ids");
    int64_t blocks = ceil_div(n_max, kBlock);
    const int64_t zero_blocks = ceil_div(n_zero_words, (int64_t)kBlock * 16) < 2048 ? ceil_div(n_zero_words, (int64_t)kBlock * 16) : 2048;
    if (blocks < zero_blocks) blocks = zero_blocks;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(idmap_insert_dst_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, stream, make_ref(d_table, slots),
                       d_dst_ids, n_max, d_n, d_uniq, d_status, d_zero_words, n_zero_words);
    FGL_CHECK_LAUNCH("idmap_insert_dst_kernel");
    return FGL_OK;
}

// the workspace of map_src: one slot index per edge, the counts of inputs too large to do without, the marks
struct IdmapScratch {
    uint32_t* slot_of;
    int32_t* line_counts;
    int32_t* tile_sums;
    int32_t* tile_prefix;
    MentionMarks marks;
    size_t used;
};
static IdmapScratch carve_idmap(void* ws, int64_t n_edges_max, bool with_marks)
{
    Carver c(ws);
    IdmapScratch o{};
    o.slot_of = c.take<uint32_t>((size_t)n_edges_max);
    o.line_counts = c.take<int32_t>((size_t)mark_tiles(n_edges_max) * (kMarkTile / kMarkLine));
    o.tile_sums = c.take<int32_t>((size_t)mark_tiles(n_edges_max));
    o.tile_prefix = c.take<int32_t>((size_t)mark_tiles(n_edges_max));
    if (with_marks) o.marks = marks_at(c.take<uint32_t>(mark_words(n_edges_max)));
    o.used = c.used();
    return o;
}

size_t idmap_map_src_workspace_bytes(int64_t n_edges_max, bool with_marks) { return carve_idmap(nullptr, n_edges_max, with_marks).used; }

InsertWork idmap_insert_work(void* d_table, int64_t slots, void* d_ws, int64_t n_edges_max, int32_t* d_src_out, const MentionMarks& marks,
                             const TransposeJob* rank_job)
{
    InsertWork w;
    w.t = make_ref(d_table, slots);
    w.slot_of = carve_idmap(d_ws, n_edges_max, false).slot_of;
    w.out = d_src_out;
    w.marks = marks;
    w.rank = rank_of(rank_job);
    return w;
}

int launch_idmap_map_src(void* d_table, int64_t slots, const int32_t* d_src_in, int32_t* d_src_out, int64_t n_edges_max,
                         const int32_t* d_n_edges, int64_t n_base, const int32_t* d_n_base, int32_t* d_n_total_out,
                         int32_t* d_uniq, int64_t uniq_capacity, int flags, uint32_t* d_status, void* d_ws,
                         size_t ws_bytes, hipStream_t stream, bool counter_is_zeroed, bool leave_table_empty,
                         const MapSrcExtras* extras)
{
    MapSrcExtras x;
    memset(&x, 0, sizeof(x));
    if (extras != nullptr) x = *extras;
    FGL_REQUIRE(d_table != nullptr && valid_slots(slots), "idmap: slot count %lld is not a power of two in [64, 2^31]", (long long)slots);
    FGL_REQUIRE((flags & ~(FGL_IDMAP_ARRIVAL | FGL_IDMAP_FINAL)) == 0, "idmap_map_src: unknown flags %d", flags);
    const bool final_call = (flags & FGL_IDMAP_FINAL) != 0;
    FGL_REQUIRE(n_edges_max >= 0 && n_base >= 0 && uniq_capacity >= 0, "idmap_map_src: negative size");
    FGL_REQUIRE(n_base + n_edges_max <= 0x7FFFFFFDll, "idmap_map_src: n_base + n_edges exceeds 31 bits");
    FGL_REQUIRE(n_edges_max == 0 || (d_src_in && d_src_out && d_uniq), "idmap_map_src: null pointer");
    FGL_REQUIRE(d_n_total_out == nullptr || d_n_total_out != d_n_base, "idmap_map_src: n_total_out must not alias n_base");
    const bool own_marks = x.marks.bits == nullptr;
    if (d_ws == nullptr || ws_bytes < idmap_map_src_workspace_bytes(n_edges_max, own_marks)) {
        set_error("idmap_map_src: workspace too small (%zu < %zu)", ws_bytes, idmap_map_src_workspace_bytes(n_edges_max, own_marks));
        return FGL_ERR_WORKSPACE;
    }
    FGL_REQUIRE(((uintptr_t)d_ws & 15) == 0, "idmap_map_src: the workspace must be 16-byte aligned");
    const int64_t tiles = mark_tiles(n_edges_max);
    const IdmapScratch ws = carve_idmap(d_ws, n_edges_max, own_marks);
    uint32_t* slot_of = ws.slot_of;
    const TableRef t = make_ref(d_table, slots);
    unsigned edge_blocks = stride_grid(n_edges_max, kBlock);
    NextHop next{};  // all null: nothing to prepare
    if (x.next_hop != nullptr) next = *x.next_hop;
    const TransposeRank tr = rank_of(x.rank_job);
    // the last pass carries steps for the transposed blocks of the hops around this one, in workgroups of their own
    // behind the pass's own
    TransposeJob scan, zero;
    memset(&scan, 0, sizeof(scan));
    memset(&zero, 0, sizeof(zero));
    ZeroJob zero_marks{};
    unsigned side_blocks = 0;
    if (x.scan_job != nullptr && x.scan_job->cnt != nullptr) {
        scan = *x.scan_job;
        scan.side_first = (int)side_blocks;
        scan.side_blocks = side_blocks_for(scan.cols_max * scan.split + 1, kTjobTile);
        side_blocks += (unsigned)scan.side_blocks;
    }
    if (x.zero_job != nullptr && x.zero_job->cnt != nullptr) {
        zero = *x.zero_job;
        zero.side_first = (int)side_blocks;
        zero.side_blocks = side_blocks_for(zero.cols_max * zero.split + 1, kBlock * 16);
        side_blocks += (unsigned)zero.side_blocks;
    }
    if (x.zero_marks.n16 > 0 && !(flags & FGL_IDMAP_ARRIVAL)) {
        zero_marks = x.zero_marks;
        zero_marks.side_first = (int)side_blocks;
        zero_marks.side_blocks = side_blocks_for(zero_marks.n16, kBlock * 4);
        side_blocks += (unsigned)zero_marks.side_blocks;
    }
    FGL_REQUIRE(!leave_table_empty || final_call, "idmap_map_src: only a final call can leave the table empty");

    if (flags & FGL_IDMAP_ARRIVAL) {
        if (x.d_dst_inout != nullptr && n_edges_max > 0) {  // (this numbering's passes do not carry the destination half: a launch of its own)
            hipLaunchKernelGGL(idmap_lookup_kernel, dim3(edge_blocks), dim3(kBlock), 0, stream, t, x.d_dst_inout, n_edges_max, d_n_edges, d_status);
            FGL_CHECK_LAUNCH("idmap_lookup_kernel");
        }
        // the counter of new ids: *d_n_total_out itself when the caller vouches that it holds zero (the all-hops
        // entry point zeroes its counts when it resets the table), else one int of the (otherwise unused)
        // prefix array, zeroed by a launch of its own
        int32_t* counter = (counter_is_zeroed && d_n_total_out) ? d_n_total_out : ws.tile_prefix;
        if (counter == ws.tile_prefix) {
            int rc0 = launch_fill_u32(reinterpret_cast<uint32_t*>(counter), 1, 0u, stream);
            if (rc0 != FGL_OK) return rc0;
        }
        if (n_edges_max > kArrivalSmallEdges)
            hipLaunchKernelGGL(idmap_insert_arrival_kernel<kArrivalItems>, dim3(stride_grid(n_edges_max, kBlock * kArrivalItems)),
                               dim3(kBlock), 0, stream, t, d_src_in,
                               n_edges_max, d_n_edges, n_base, d_n_base, slot_of, counter, d_uniq, uniq_capacity, d_src_out,
                               d_status, next, tr);
        else
            hipLaunchKernelGGL(idmap_insert_arrival_kernel<1>, dim3(edge_blocks), dim3(kBlock), 0, stream, t, d_src_in,
                               n_edges_max, d_n_edges, n_base, d_n_base, slot_of, counter, d_uniq, uniq_capacity, d_src_out,
                               d_status, next, tr);
        FGL_CHECK_LAUNCH("idmap_insert_arrival_kernel");
        hipLaunchKernelGGL(idmap_relabel_publish_kernel, dim3(edge_blocks + side_blocks), dim3(kBlock), 0, stream, t, n_edges_max, d_n_edges,
                           slot_of, d_src_out, counter, n_base, d_n_base, uniq_capacity, d_n_total_out, d_status, tr, scan, zero, x.d_readback,
                           x.d_readback_counts, x.n_readback_counts);
        FGL_CHECK_LAUNCH("idmap_relabel_publish_kernel");
    } else {
        MentionMarks marks = x.marks;
        if (own_marks) {  // (nobody has cleared them)
            marks = ws.marks;
            int rc0 = launch_fill_u32(reinterpret_cast<uint32_t*>(marks.bits), (int64_t)mark_words(n_edges_max), 0u, stream);
            if (rc0 != FGL_OK) return rc0;
        }
        if (!x.inserted) {
            const InsertWork w = idmap_insert_work(d_table, slots, d_ws, n_edges_max, d_src_out, marks, x.rank_job);
            hipLaunchKernelGGL(idmap_insert_src_kernel, dim3(edge_blocks), dim3(kBlock), 0, stream, d_src_in, n_edges_max, d_n_edges, w,
                               d_status, x.d_dst_inout);
            FGL_CHECK_LAUNCH("idmap_insert_src_kernel");
        }
#define FGL_LAUNCH_NUMBER(MODE, WB, TILES, TOTAL, STATUS, READBACK)                                                              \
    hipLaunchKernelGGL((idmap_number_kernel<MODE, WB>), dim3(edge_blocks + side_blocks), dim3(kBlock), 0, stream, t, d_src_in,    \
                       n_edges_max, d_n_edges, n_base, d_n_base, slot_of, marks, ws.line_counts, TILES, d_uniq, uniq_capacity,      \
                       d_src_out, TOTAL, STATUS, next, tr, scan, zero, zero_marks, (int)side_blocks, READBACK, x.d_readback_counts, \
                       x.n_readback_counts)
        const bool from_bits = n_edges_max <= (int64_t)kLinesInLds * kMarkLine;
        if (!from_bits) {
            const int64_t count_blocks = ceil_div(tiles * (kMarkTile / kMarkLine), kBlock);
            hipLaunchKernelGGL(idmap_count_kernel, dim3((unsigned)(count_blocks < 2048 ? count_blocks : 2048)), dim3(kBlock), 0, stream, marks,
                               n_edges_max, d_n_edges, ws.line_counts, ws.tile_sums);
            FGL_CHECK_LAUNCH("idmap_count_kernel");
        }
        // every workgroup of a pass that scans the counts itself pays for that scan once: a few workgroups per
        // compute unit, each looping over several tiles of edges, instead of one per 256 edges
        if (tiles <= kLinesInLds) {
            if (edge_blocks > kNumberMaxBlocks) edge_blocks = kNumberMaxBlocks;
            if (from_bits && final_call) FGL_LAUNCH_NUMBER(kFromBits, false, nullptr, d_n_total_out, d_status, x.d_readback);
            else if (from_bits) FGL_LAUNCH_NUMBER(kFromBits, true, nullptr, d_n_total_out, d_status, x.d_readback);
            else if (final_call) FGL_LAUNCH_NUMBER(kFromTiles, false, ws.tile_sums, d_n_total_out, d_status, x.d_readback);
            else FGL_LAUNCH_NUMBER(kFromTiles, true, ws.tile_sums, d_n_total_out, d_status, x.d_readback);
        } else {
            hipLaunchKernelGGL(idmap_prefix_publish_kernel, dim3(1), dim3(1024), 0, stream, ws.tile_sums, ws.tile_prefix, n_edges_max,
                               d_n_edges, n_base, d_n_base, uniq_capacity, d_n_total_out, d_status, x.d_readback, x.d_readback_counts,
                               x.n_readback_counts);
            FGL_CHECK_LAUNCH("idmap_prefix_publish_kernel");
            if (final_call) FGL_LAUNCH_NUMBER(kFromPrefix, false, ws.tile_prefix, nullptr, nullptr, nullptr);
            else FGL_LAUNCH_NUMBER(kFromPrefix, true, ws.tile_prefix, nullptr, nullptr, nullptr);
        }
#undef FGL_LAUNCH_NUMBER
        FGL_CHECK_LAUNCH("idmap_number_kernel");
    }
    // (the last pass reads the table: emptying it takes a launch of its own)
    if (leave_table_empty) return launch_idmap_reset(d_table, slots, stream);
    return FGL_OK;
}

}  // namespace fgl

using namespace fgl;

FGL_EXPORT int64_t fgl_table_size(int64_t num, int scale)
{
    // (largest power of two <= num) << scale, as cuda_hashtable.cuh:27-30 computes for num >= 2
    int64_t half = num >> 1, p = 1;
    if (half >= 1) {
        int lg = 0;
        while ((half >> (lg + 1)) != 0) ++lg;
        p = (int64_t)1 << (1 + lg);
    }
    return p << scale;
}

FGL_EXPORT int64_t fgl_idmap_slots(int64_t max_unique)
{
    int64_t want = 2 * (max_unique > 0 ? max_unique : 0);
    int64_t s = 64;
    while (s < want) s <<= 1;
    return s;
}

FGL_EXPORT size_t fgl_idmap_table_bytes(int64_t slots) { return slots > 0 ? (size_t)slots * 8 : 0; }

FGL_EXPORT int fgl_idmap_reset(void* d_table, int64_t slots, void* stream) { return launch_idmap_reset(d_table, slots, as_stream(stream)); }

FGL_EXPORT int fgl_idmap_insert_dst(void* d_table, int64_t slots, const int32_t* d_dst_ids, int64_t n_max,
                                    const int32_t* d_n, int32_t* d_uniq, uint32_t* d_status, void* stream)
{
    return launch_idmap_insert_dst(d_table, slots, d_dst_ids, n_max, d_n, d_uniq, d_status, as_stream(stream), nullptr, 0);
}

FGL_EXPORT size_t fgl_idmap_map_src_workspace_bytes(int64_t n_edges_max) { return idmap_map_src_workspace_bytes(n_edges_max < 0 ? 0 : n_edges_max, true); }

FGL_EXPORT int fgl_idmap_map_src(void* d_table, int64_t slots, const int32_t* d_src_in, int32_t* d_src_out,
                                 int64_t n_edges_max, const int32_t* d_n_edges, int64_t n_base, const int32_t* d_n_base,
                                 int32_t* d_n_total_out, int32_t* d_uniq, int64_t uniq_capacity, int flags,
                                 uint32_t* d_status, void* d_ws, size_t ws_bytes, void* stream)
{
    const bool leave_empty = (flags & FGL_IDMAP_LEAVE_TABLE_EMPTY) != 0;
    FGL_REQUIRE(!leave_empty || (flags & FGL_IDMAP_FINAL), "idmap_map_src: FGL_IDMAP_LEAVE_TABLE_EMPTY needs FGL_IDMAP_FINAL");
    return launch_idmap_map_src(d_table, slots, d_src_in, d_src_out, n_edges_max, d_n_edges, n_base, d_n_base,
                                d_n_total_out, d_uniq, uniq_capacity, flags & ~FGL_IDMAP_LEAVE_TABLE_EMPTY, d_status, d_ws, ws_bytes,
                                as_stream(stream), false, leave_empty, nullptr);
}

FGL_EXPORT int fgl_idmap_transfer(void* d_table, int64_t slots, const int32_t* d_dst_unique, int64_t n_dst,
                                  int32_t* d_src_edges, int32_t* d_dst_edges, int64_t n_edges, int32_t* d_uniq,
                                  int64_t uniq_capacity, int flags, int32_t* d_n_total_out, uint32_t* d_status,
                                  int32_t* d_readback, void* d_ws, size_t ws_bytes, void* stream)
{
    FGL_REQUIRE(n_dst >= 0 && n_edges >= 0, "idmap_transfer: negative size");
    FGL_REQUIRE(n_edges == 0 || (d_src_edges && d_dst_edges), "idmap_transfer: null edge array");
    FGL_REQUIRE(d_src_edges == nullptr || d_src_edges != d_dst_edges, "idmap_transfer: the two edge arrays must be distinct");
    FGL_REQUIRE(d_uniq != nullptr && uniq_capacity >= n_dst, "idmap_transfer: the unique list cannot hold the destination ids");
    const bool leave_empty = (flags & FGL_IDMAP_LEAVE_TABLE_EMPTY) != 0;
    FGL_REQUIRE(!leave_empty || (flags & FGL_IDMAP_FINAL), "idmap_transfer: FGL_IDMAP_LEAVE_TABLE_EMPTY needs FGL_IDMAP_FINAL");
    if (d_ws == nullptr || ws_bytes < idmap_map_src_workspace_bytes(n_edges, true)) {
        set_error("idmap_transfer: workspace too small (%zu < %zu)", ws_bytes, idmap_map_src_workspace_bytes(n_edges, true));
        return FGL_ERR_WORKSPACE;
    }
    FGL_REQUIRE(((uintptr_t)d_ws & 15) == 0, "idmap_transfer: the workspace must be 16-byte aligned");
    // the marks of the source ids' first mentions are cleared by the launch that inserts the destination ids
    MapSrcExtras x;
    memset(&x, 0, sizeof(x));
    x.marks = carve_idmap(d_ws, n_edges, true).marks;
    x.d_dst_inout = d_dst_edges;
    x.d_readback = d_readback;
    int rc = launch_idmap_insert_dst(d_table, slots, d_dst_unique, n_dst, nullptr, d_uniq, d_status, as_stream(stream),
                                     reinterpret_cast<uint32_t*>(x.marks.bits), (int64_t)mark_words(n_edges));
    if (rc != FGL_OK) return rc;
    return launch_idmap_map_src(d_table, slots, d_src_edges, d_src_edges, n_edges, nullptr, n_dst, nullptr, d_n_total_out, d_uniq,
                                uniq_capacity, flags & ~FGL_IDMAP_LEAVE_TABLE_EMPTY, d_status, d_ws, ws_bytes, as_stream(stream), false,
                                leave_empty, &x);
}

FGL_EXPORT int fgl_idmap_lookup(const void* d_table, int64_t slots, int32_t* d_ids, int64_t n_max, const int32_t* d_n,
                                uint32_t* d_status, void* stream)
{
    FGL_REQUIRE(d_table != nullptr && valid_slots(slots), "idmap: slot count %lld is not a power of two in [64, 2^31]", (long long)slots);
    FGL_REQUIRE(n_max >= 0, "idmap_lookup: negative size");
    if (n_max == 0) return FGL_OK;
    FGL_REQUIRE(d_ids != nullptr, "idmap_lookup: null ids");
    hipLaunchKernelGGL(idmap_lookup_kernel, dim3(stride_grid(n_max, kBlock)), dim3(kBlock), 0, as_stream(stream),
                       make_ref(const_cast<void*>(d_table), slots), d_ids, n_max, d_n, d_status);
    FGL_CHECK_LAUNCH("idmap_lookup_kernel");
    return FGL_OK;
}
