// Which row of a CSR every entry of a tile belongs to, for passes that deal the entries out evenly whatever the rows' lengths
// (a hub's row walked by one lane group outlasts everything else: 54 M entries with rows of up to 85 K took 21 ms that way).
// Two steps: a pass over the rows notes the row that holds each tile's first entry (mark_tile_rows); the tile's workgroup marks
// the rows that begin inside it and spreads the marks by a running maximum (tile_rows).
#pragma once
#include "fgl_common.hpp"

namespace fgl {

#if defined(__HIPCC__)

// row r names the tiles that begin inside it.  Row 0 also names those in front of its first entry (offsets that do not start at
// zero, as a slice of a larger CSR has them): tile_rows reads the entry of every tile below the last offset and goes by it.
template <int TILE>
__device__ __forceinline__ void mark_tile_rows(const int32_t* __restrict__ indptr, int64_t r, int64_t tiles, int32_t* __restrict__ tile_row)
{
    int64_t a = indptr[r];
    const int64_t b = indptr[r + 1];
    if (r == 0 || a < 0) a = 0;
    for (int64_t t = (a + TILE - 1) / TILE; t * TILE < b && t < tiles; ++t) tile_row[t] = (int32_t)r;
}

// s_row[i] = row of entry tile * TILE + i, for the entries below n (TILE = NT * ITEMS; ITEMS a multiple of four; s_row 16-byte
// aligned; s_wave: NT / 64 ints).  Barriers: every thread of the workgroup must call it.
template <int NT, int ITEMS>
__device__ __forceinline__ void tile_rows(const int32_t* __restrict__ indptr, int64_t n_rows, const int32_t* __restrict__ tile_row,
                                          int64_t tile, int64_t n, int* s_row, int* s_wave)
{
    constexpr int kTile = NT * ITEMS;
    const int64_t e0 = tile * kTile;
    const bool any = e0 < n, more = e0 + kTile < n;
    const int64_t r0 = any ? tile_row[tile] : 0;
    const int64_t r1 = more ? tile_row[tile + 1] : n_rows - 1;  // the last row that may begin in the tile
    if (any && r1 - r0 > 4 * kTile) {
        // a gap of empty rows far longer than the tile: every entry looks its row up (the last row that begins at or before it)
        for (int i = (int)threadIdx.x; i < kTile && e0 + i < n; i += NT) {
            int64_t lo = r0, hi = r1 + 1;  // indptr[lo] <= e < indptr[hi]
            while (hi - lo > 1) {
                const int64_t mid = (lo + hi) >> 1;
                if (indptr[mid] <= e0 + i) lo = mid; else hi = mid;
            }
            s_row[i] = (int)lo;
        }
        __syncthreads();
        return;
    }
    int4* v4 = reinterpret_cast<int4*>(s_row) + (int)threadIdx.x * (ITEMS / 4);
#pragma unroll
    for (int q = 0; q < ITEMS / 4; ++q) v4[q] = make_int4(0, 0, 0, 0);
    __syncthreads();
    if (any) {
        if (threadIdx.x == 0) s_row[0] = (int)r0;
        for (int64_t r = r0 + 1 + threadIdx.x; r <= r1; r += NT) {
            const int64_t a = indptr[r], b = indptr[r + 1];
            if (b > a && a > e0 && a < e0 + kTile) s_row[a - e0] = (int)r;  // (rows with entries begin at distinct places)
        }
    }
    __syncthreads();
    int v[ITEMS];
#pragma unroll
    for (int q = 0; q < ITEMS / 4; ++q) {
        const int4 x = v4[q];
        v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
    }
#pragma unroll
    for (int j = 1; j < ITEMS; ++j) v[j] = v[j] > v[j - 1] ? v[j] : v[j - 1];
    int top = v[ITEMS - 1];
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int o = __shfl_up(top, d, kWave);
        if (lane_id() >= d && o > top) top = o;
    }
    if (lane_id() == kWave - 1) s_wave[threadIdx.x / kWave] = top;
    int before = __shfl_up(top, 1, kWave);
    if (lane_id() == 0) before = 0;
    __syncthreads();
    for (int w = 0; w < (int)(threadIdx.x / kWave); ++w) before = s_wave[w] > before ? s_wave[w] : before;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) v[j] = v[j] > before ? v[j] : before;
#pragma unroll
    for (int q = 0; q < ITEMS / 4; ++q) v4[q] = make_int4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
    __syncthreads();
}

#endif  // __HIPCC__

}  // namespace fgl
