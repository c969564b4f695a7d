// Device helpers of the id-map passes (fgl_idmap.hip): an edge's insert into the table, and what a newly numbered
// node hands to the next hop's sampling.
#pragma once
#include "fgl_common.hpp"
#include "fgl_kernels.hpp"
#include "fgl_table.hpp"
#include "fgl_transpose_job.hpp"

namespace fgl {

// what a launch needs to insert the ids of a hop's edges (idmap_insert_src_kernel, the sampling kernels)
struct InsertWork {
    TableRef t;
    uint32_t* slot_of;  // per edge: the id's slot; kDone: relabelled already; kEmpty: no slot
    int32_t* out;       // the edges' local ids
    MentionMarks marks;
    TransposeRank rank;
};

#if defined(__HIPCC__)

// find_or_insert for an edge's source id, which also says what becomes of the marks:
// *holder = this edge became the first known mention of the id (it installed the key, or lowered
// the key's first-edge index to its own); *displaced = the pending value it took that place from (kEmpty: none).
// An edge that became holder and is never displaced is the id's first mention.
// The probe sequence is entered at slot p with that slot's value already in hand (`s`: loaded, or returned by a
// failed compare-and-swap), so that a caller can have the first loads -- and the first compare-and-swaps -- of
// several edges in flight together before it walks any sequence further.
__device__ __forceinline__ uint32_t insert_mention_from(const TableRef t, uint32_t id, uint32_t mine, uint32_t p,
                                                        unsigned long long s, uint32_t* seen_val, bool* holder,
                                                        uint32_t* displaced)
{
    unsigned long long* slots = reinterpret_cast<unsigned long long*>(t.words);
    const unsigned long long fresh = (unsigned long long)id | ((unsigned long long)mine << 32);
    const uint32_t limit = t.mask < kMaxProbes ? t.mask + 1 : kMaxProbes;
    *holder = false;
    *displaced = kEmpty;
    for (uint32_t n = 0; n < limit; ++n) {
        if ((uint32_t)s == kEmpty) {
            const unsigned long long seen = atomicCAS(&slots[p], ~0ull, fresh);
            if (seen == ~0ull) {
                *seen_val = mine;
                *holder = true;
                return p;
            }
            s = seen;
        }
        if ((uint32_t)s == id) {
            const uint32_t v = (uint32_t)(s >> 32);
            *seen_val = v;
            if ((v & kPending) && v > mine) {
                const uint32_t old = atomicMin(&t.words[2 * (size_t)p + 1], mine);
                if (old > mine) {  // (else an even earlier mention got there between the load and the atomic)
                    *holder = true;
                    *displaced = old;
                }
            }
            return p;
        }
        p = (p + 1) & t.mask;
        s = slots[p];
    }
    return kEmpty;
}

// What is left of edge e's insert once its slot is known (q; kEmpty: none found): the slot is noted for the number pass, or the
// edge relabelled here and now; the edge whose place it took loses its mark.  n_e bounds the indices that marks exist for.
__device__ __forceinline__ void finish_insert(const InsertWork& w, int64_t e, int64_t n_e, int32_t id, uint32_t q, uint32_t seen,
                                              uint32_t displaced, uint32_t* __restrict__ d_status)
{
    if (q == kEmpty) {
        // table full, or not a node id: reported; the edge's local id becomes -1 (written by the number pass)
        if (d_status) atomicOr(d_status, id >= 0 ? FGL_STATUS_TABLE_FULL : FGL_STATUS_BAD_ID);
    } else if (!(seen & kPending)) {
        // numbered in an earlier hop (or a destination node): the edge is relabelled right here and
        // takes no further part (`out` may be the array the id came from: this lane is the only one that touches entry e)
        w.out[e] = (int32_t)seen;
        take_rank(w.rank, e, (int32_t)seen);
        q = kDone;
    } else if (displaced != kEmpty) {
        // (an edge of this hop: ids of earlier hops hold their local id, or all ones if the unique list had no room for them.
        // The bound only matters to a caller that goes on with a table which a final call has left unnumbered.)
        const int64_t d = (int64_t)(displaced & ~kPending);
        if (d < n_e) atomicXor(&w.marks.bits[d >> 6], 1ull << (d & 63));
    }
    w.slot_of[e] = q;
}

// The marks of the wave's edges that became holders: lane l's edge is first + l.  Every lane of the wave calls it.
__device__ __forceinline__ void mark_first(const MentionMarks& m, int64_t first, bool holder)
{
    const unsigned long long won = __ballot(holder);
    const int lane = lane_id(), off = (int)(first & 63);
    if (lane == 0 && (won << off) != 0) atomicXor(&m.bits[first >> 6], won << off);
    if (lane == 1 && off != 0 && (won >> (64 - off)) != 0) atomicXor(&m.bits[(first >> 6) + 1], won >> (64 - off));
}

// marks of a line of edges, and of its edges before edge ef (final once every insert of the hop is done)
__device__ __forceinline__ int line_count(const MentionMarks& m, int64_t line)
{
    const ulonglong2* w = reinterpret_cast<const ulonglong2*>(m.bits + line * (kMarkLine / 64));
    const ulonglong2 w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];
    return __popcll(w0.x) + __popcll(w0.y) + __popcll(w1.x) + __popcll(w1.y) + __popcll(w2.x) + __popcll(w2.y) + __popcll(w3.x) + __popcll(w3.y);
}
__device__ __forceinline__ int marks_before_in_line(const MentionMarks& m, int64_t ef)
{
    const ulonglong2* w = reinterpret_cast<const ulonglong2*>(m.bits + ef / kMarkLine * (kMarkLine / 64));
    const ulonglong2 w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3];
    const int word = (int)(ef >> 6) & 7;
    const unsigned long long bits[8] = {w0.x, w0.y, w1.x, w1.y, w2.x, w2.y, w3.x, w3.y};
    const unsigned long long below = (1ull << (ef & 63)) - 1ull;
    int n = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) n += __popcll(j < word ? bits[j] : j == word ? bits[j] & below : 0ull);
    return n;
}

// A node that has just been given a position in the unique list is a seed of the next hop: its row start and
// degree go to that position (store_next_hop), and its min(fanout, degree) to the next hop's per-tile edge counts.
// The two graph offsets are read by load_row_of, which callers issue early -- for every edge that may turn out to
// be a first mention -- so that the reads overlap the pass's own chain of loads.  An id outside the graph is
// marked for the next hop's sampling kernel to report.
__device__ __forceinline__ void load_row_of(const NextHop& next, int32_t id, int64_t* a, int64_t* deg)
{
    *a = kRowBadId;
    *deg = 0;
    if (id >= 0 && (int64_t)id < next.n_nodes) {
        if (next.is64) {
            const int64_t* p = static_cast<const int64_t*>(next.indptr);
            *a = p[id];
            *deg = p[id + 1] - *a;
        } else {
            const int32_t* p = static_cast<const int32_t*>(next.indptr);
            *a = p[id];
            *deg = (int64_t)p[id + 1] - *a;
        }
        if (*deg < 0) *deg = 0;
        if (*deg > 0x7FFFFFFF) *deg = 0x7FFFFFFF;
    }
}

__device__ __forceinline__ int store_next_hop(const NextHop& next, int64_t local, int64_t a, int64_t deg)
{
    next.row_start[local] = a;
    next.deg[local] = (int32_t)deg;
    return deg < next.fanout ? (int)deg : next.fanout;
}

#endif  // __HIPCC__

}  // namespace fgl
