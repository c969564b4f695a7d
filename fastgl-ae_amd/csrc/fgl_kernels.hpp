// Internal launchers shared between the translation units of libfastgl_hip.
#pragma once
#include "fgl_common.hpp"

namespace fgl {

// exclusive sum (fgl_scan.hip).  d_out gets n+1 entries; d_total_extra (optional) the total.
size_t scan_workspace_bytes(int64_t n_max);
int launch_exclusive_sum(const int32_t* d_in, int64_t n_max, const int32_t* d_n, int32_t* d_out,
                         int32_t* d_total_extra, void* d_ws, size_t ws_bytes, hipStream_t stream);
// single-workgroup scan of per-tile sums; the total is written to *total_a, *total_b and
// at_count_base[actual count of (n_max, d_n)] (each optional); tile_items > 0 restricts the
// scan to the tiles the actual count occupies
int launch_tile_prefix(const int32_t* tile_sums, int n_tiles, int32_t* tile_prefix, int32_t* total_a,
                       int32_t* total_b, int32_t* at_count_base, int64_t n_max, const int32_t* d_n, int tile_items,
                       hipStream_t stream, int32_t* readback = nullptr, const uint32_t* d_status = nullptr);
int launch_fill_u32(uint32_t* p, int64_t n, uint32_t value, hipStream_t stream);

// which kernel the calling thread's last dense product was formed by (fgl_product_last_kernel)
void note_product(const char* kernel);

// Row start of a node whose id lies outside the graph / whose insert found the table full: how a launch that
// must not touch the status word hands the error to the next one that reads the entry.
constexpr int64_t kRowBadId = -1;
constexpr int64_t kRowTableFull = -2;

// What a pass over a hop's nodes prepares for the sampling of the next hop: row start and degree of every node
// at its position in the unique list, and the per-tile sums of min(fanout, degree) that place the tiles' output.
struct NextHop {
    const void* indptr;
    int is64;
    int64_t n_nodes;
    int64_t* row_start;
    int32_t* deg;
    int32_t* tile_sums;  // zeroed by the caller; [position / tile_seeds] += min(fanout, degree)
    int fanout;
    int tile_seeds;
};

// A block's transposed form under construction inside the all-hops call (fgl_transpose_job.hpp).  cnt == nullptr:
// no such work.
struct TransposeJob {
    int32_t* cnt;        // split * cols_max + 1 counters, then their prefix sums; split == 1: the same array as t_ptr
    int32_t* tile_sums;  // one per 2048 counters
    int32_t* rank;       // per edge: its position within its transposed row
    int32_t* t_ptr;      // cols_max + 1
    int32_t* t_dst;      // edges_max
    int32_t* t_edge;     // edges_max, or null
    int32_t* longest;    // one int, zero before the scan step: the longest transposed row if beyond FGL_SHORT_ROW_ENTRIES
    const int32_t* block_ptr;
    const int32_t* src_local;
    const int32_t* d_n_rows;
    const int32_t* d_n_cols;
    const int32_t* d_n_edges;
    int64_t rows_max, cols_max, edges_max;
    int split;
    // which workgroups of the launch at hand work on the step it carries: side_blocks of them, the last of the
    // grid but side_first (set per launch by the launcher, which appends them to the grid)
    int side_blocks, side_first;
};
// Side workgroups for a step over n_items, items_per_block at a time: never more than the work needs, and few
// enough that they are an appendix to the launch that carries them.
inline int side_blocks_for(int64_t n_items, int64_t items_per_block, int cap = 8192)
{
    int64_t b = (n_items + items_per_block - 1) / items_per_block;
    if (b < 1) b = 1;
    return (int)(b < cap ? b : cap);
}
// what the id-map passes need of it: where an edge takes its rank
struct TransposeRank {
    int32_t* cnt;
    int32_t* rank;  // null: no transposed block is being built
    int64_t cols_max;
    int split;
};
__host__ __device__ inline TransposeRank rank_of(const TransposeJob* j)
{
    return j && j->cnt ? TransposeRank{j->cnt, j->rank, j->cols_max, j->split} : TransposeRank{nullptr, nullptr, 0, 1};
}
// what a hop's sampling launch carries along for the transposed blocks of the hops before it: the tile sums of the last hop's
// counters, the filling of the rows of the hop before that
struct TransposeSteps {
    TransposeJob sums;
    TransposeJob fill;
};
// memory to clear in side workgroups of a launch
struct ZeroJob {
    uint4* p;
    int64_t n16;  // 16-byte pieces; 0: no such work
    int side_blocks, side_first;
};

// Which edges of a hop are the first mentions of new ids, kept exact while the ids are being inserted: a bit per edge, changed
// with commutative integer atomics only (fgl_idmap_device.hpp), so that an edge can be marked by its own wave and unmarked by
// whoever finds an earlier mention, in either order; when the last insert is done they are the final state.  All zero before the
// first insert of a hop.
constexpr int kMarkLine = 512;   // edges whose bits are one 64-byte line
constexpr int kMarkTile = 4096;  // edges per entry of the scanned counts of large hops: eight lines
struct MentionMarks {
    unsigned long long* bits;
};
__host__ __device__ inline int64_t mark_tiles(int64_t n_edges) { return n_edges > 0 ? (n_edges + kMarkTile - 1) / kMarkTile : 1; }
inline size_t mark_words(int64_t n_edges) { return (size_t)mark_tiles(n_edges) * (kMarkTile / 32); }  // 32-bit words, a multiple of 4
inline MentionMarks marks_at(uint32_t* words) { return MentionMarks{reinterpret_cast<unsigned long long*>(words)}; }

// neighbour sampling (fgl_sample.hip)
int sample_tile_seeds(int fanout, int64_t n_seeds_max);      // seeds per tile of the per-hop operator ...
int sample_hop_tile_seeds(int fanout, int64_t n_seeds_max);  // ... and of a mini-batch's hops
int64_t sample_tile_count(int64_t n_seeds_max, int fanout);
size_t sample_workspace_bytes(int64_t n_seeds_max, int fanout);
// the second half of launch_sample, for callers that hold row starts, degrees and tile sums already
struct InsertWork;
bool sample_can_insert(int fanout, int64_t n_seeds_max);  // the launch can put the ids it samples into the id-map's table itself
int launch_sample_edges(const int32_t* d_indices, const int32_t* d_seeds, int64_t n_seeds_max, const int32_t* d_n_seeds,
                        int fanout, const int64_t* row_start, const int32_t* deg, const int32_t* tile_sums,
                        int32_t* tile_prefix, uint64_t rng_seed, uint32_t stream_id, int32_t* d_src_out,
                        int32_t* d_dst_out, int32_t* d_block_ptr, int32_t* d_n_edges_out, uint32_t* d_status,
                        hipStream_t stream, const uint32_t* d_stream_add, const NextHop* next,
                        const TransposeSteps* steps,             // (optional) steps for the transposed blocks of earlier hops
                        int32_t* d_readback,                     // (optional) {edge count, status word} once both are final; may be host memory
                        const InsertWork* insert,                // (optional, where sample_can_insert) insert the sampled ids
                        int tile_seeds);                         // seeds per entry of tile_sums: sample_hop_tile_seeds / sample_tile_seeds
int launch_sample(const void* d_indptr, int indptr_is64, const int32_t* d_indices, int64_t n_nodes,
                  const int32_t* d_seeds, int64_t n_seeds_max, const int32_t* d_n_seeds, int fanout,
                  uint64_t rng_seed, uint32_t stream_id, int32_t* d_src_out, int32_t* d_dst_out,
                  int32_t* d_block_ptr, int32_t* d_n_edges_out, uint32_t* d_status, void* d_ws, size_t ws_bytes,
                  hipStream_t stream, const uint32_t* d_stream_add = nullptr, int32_t* d_readback = nullptr);

// id-map (fgl_idmap.hip)
size_t idmap_map_src_workspace_bytes(int64_t n_edges_max, bool with_marks);  // with_marks: the marks live there too
int launch_idmap_reset(void* d_table, int64_t slots, hipStream_t stream);
int launch_idmap_insert_dst(void* d_table, int64_t slots, const int32_t* d_dst_ids, int64_t n_max,
                            const int32_t* d_n, int32_t* d_uniq, uint32_t* d_status, hipStream_t stream,
                            uint32_t* d_zero_words, int64_t n_zero_words);  // (optional) scratch words to clear on the way
// what the callers inside the library add to map_src (all optional)
struct MapSrcExtras {
    MentionMarks marks;          // cleared already; bits == null: the call clears and uses marks of its own, in its workspace
    bool inserted;               // the sampling launch has inserted the edges' ids (idmap_insert_work): only the number pass is left
    const NextHop* next_hop;     // the new nodes are seeds of a next hop: prepare its sampling
    const TransposeJob* rank_job;  // the edges take their ranks in this block's transposed rows
    const TransposeJob* scan_job;  // scan step of the hop before, carried by the last pass
    const TransposeJob* zero_job;  // the next hop's counters, cleared by the last pass
    ZeroJob zero_marks;            // the next hop's marks, cleared by the last pass (first-occurrence order only)
    int32_t* d_dst_inout;          // n_edges_max ids that are in the table already: relabelled in place by the first pass
    int32_t* d_readback;           // {node total, status word} once both are final; may be host memory
    const int32_t* d_readback_counts;  // instead of those two words: a copy of this array, which holds *d_n_total_out and
    int n_readback_counts;             //   the status word, taken when the node total is final
};
int launch_idmap_map_src(void* d_table, int64_t slots, const int32_t* d_src_in, int32_t* d_src_out,
                         int64_t n_edges_max, const int32_t* d_n_edges, int64_t n_base, const int32_t* d_n_base,
                         int32_t* d_n_total_out, int32_t* d_uniq, int64_t uniq_capacity, int flags,
                         uint32_t* d_status, void* d_ws, size_t ws_bytes, hipStream_t stream,
                         bool counter_is_zeroed,          // arrival order: *d_n_total_out holds zero and may count the new ids
                         bool leave_table_empty,          // final calls only: every slot of the table is empty when the call's work is done
                         const MapSrcExtras* extras);
InsertWork idmap_insert_work(void* d_table, int64_t slots, void* d_ws, int64_t n_edges_max, int32_t* d_src_out, const MentionMarks& marks,
                             const TransposeJob* rank_job);

// counting and transpose of large inputs (fgl_bucket.hip)
size_t count_workspace_bytes(int64_t n_ids, int64_t n_counters);  // 0: counted with atomics, no workspace
bool launch_count(const int32_t* d_ids, int64_t n_ids, const int32_t* d_n, int64_t n_counters, int32_t* d_counts, void* d_ws,
                  hipStream_t stream, int* rc);
bool bucket_transpose_form(int64_t n_entries, int64_t n_cols);
size_t bucket_workspace_bytes(int64_t n_entries, int64_t n_cols, bool rows, bool edges);
int launch_bucket_transpose(const int32_t* d_indptr, const int32_t* d_indices, int64_t n_rows, int64_t n_cols, int64_t n_edges,
                            int32_t* d_t_indptr, int32_t* d_t_indices, int32_t* d_t_edge, int32_t* d_longest, void* d_ws, hipStream_t stream);

// deterministic block transpose (fgl_transpose_sort.hip): fills t_indices / t_edge given the offsets
size_t sorted_transpose_workspace_bytes(int64_t n_cols, int64_t n_edges);
int launch_sorted_transpose_fill(const int32_t* d_indptr, const int32_t* d_indices, int64_t n_rows, int64_t n_cols,
                                 int64_t n_edges, int32_t* d_t_indices, int32_t* d_t_edge, void* d_ws, size_t ws_bytes,
                                 hipStream_t stream);

}  // namespace fgl
