// Weight gradient of a dense layer: C[m, n] = sum over k of A[k, m] * B[k, n], both operands row-major with the long
// dimension k outermost (A = the layer's input rows, B = the gradient of its output rows; the reference forms it with
// torch::mm on a transposed view, cuda_operators/aggregate_acc.cpp:371-374,402-405).  k is the node count of a block --
// 10^4 .. 10^6 -- and C is a few hundred columns square, so there are only a handful of output tiles and the chip is
// filled by splitting k.
//
// What bounds it: in fp32 the matrix cores (157 TFLOP/s dense; 2.5 M x 100 x 64 takes 0.2 ms) and the one pass over A and
// B about equally; in bf16 the pass over A and B.
//
// Tile: a wave holds (32 VA) x (32 VB) outputs in its accumulators, VA, VB in {1, 2, 4}.  No operand goes through LDS: with
// k outermost a row of A *is* the matrix instruction's operand -- 32 lanes, one column each -- and since the order of the
// output columns inside a tile is free, lane i takes the VA neighbouring columns VA i .. VA i + VA - 1 with one vector load and
// feeds them to VA different instructions.  fp32: one row per half-wave (v_mfma_f32_32x32x2_f32 has k = 2).  bf16:
// eight rows per half-wave (v_mfma_f32_32x32x16_bf16 wants eight consecutive k per lane), turned from row pairs into
// k pairs by one v_perm per two elements.  The next rows are in flight while the current ones are multiplied.
// The four waves of a workgroup take every fourth group of rows, their accumulators are added through LDS, and
// the workgroup's sum goes to scratch; a second launch adds the k splits in a fixed order (the same bits on every run)
// and stores C in the operands' type.
// Workgroups that work on the same rows (different tiles of C) are neighbours on one XCD: the rows come from its L2 for all
// but the first of them.
//
// Measured (launch pair, MI355X; the library GEMM on the transposed view before it): fp32 100 x 256, k = 105 K: 190 -> 72 us
// (the padded products alone take 45 us at the 154 TFLOP/s a large fp32 GEMM reaches, the sum over the splits and the two
// launches about 15); 100 x 64, k = 2.4 M: 3318 -> 465 us (products alone 300, loads alone 280: the two overlap by half);
// 602 x 256, k = 8192: 57 -> 42 us; bf16 100 x 256, k = 105 K: 245 -> 25 us, 100 x 64, k = 2.4 M: 2745 -> 148 us (5.3 TB/s).
// Eight rows a step and one step ahead: 16 and 24 rows measured the same within 3 %.
//
// The split form of fp32: the fp32 matrix instructions' rate is what the wide tiles wait for, and their 256 accumulators a lane
// leave one wave a SIMD, which nothing covers while it waits for rows.  Each value is three bf16 parts instead, a product six
// bf16 products (fgl_split_product.hip says which and how exact that is), in tiles of 64 x 64, two waves a SIMD: one splits (88
// instructions for a step's 64 columns) while the other multiplies.  Every step's products are added up from zero before they are
// added to the accumulators; and since what a matrix instruction cuts off is cut downwards, which over 10^4 .. 10^6 rows adds up
// (7e-7 of the result's 2-norm for k = 107 K where the fp32 form has 2.8e-7), every other step is formed of A's negative and
// subtracted: 1.4e-7. us, fp32 / split: 100 x 256 k = 107 K 68 / 65, k = 16 K 33 / 21, k = 2000 26 / 12; 256 x 256 k = 17 K 36 /
// 29, k = 5000 31 / 16; 128 x 128 k = 60 K 37 / 28; 602 x 256 k = 8192 41 / 38; 256 x 47 k = 20 K 19 / 16.  Waves that meet
// values of which bits are lost to a result, or results that are no numbers, form their rows again (one column of the first of
// these at 1e-36: 121).  What it waits for now is the rows: one step ahead is half a microsecond at these rates. Tried: blocks of
// 128 x 128 through LDS, in which every value is split once (65 us for the first of these, but 34 and 41 for 256 x 256 and 602 x
// 256), and two steps ahead, for which the registers do not suffice (89).
//
// A lane whose columns would leave the row takes the row's last VA columns instead (its sums are then bit-equal copies of
// its neighbour's); rows past the end are replaced by zeros.  No access leaves the operands.
#include "fgl_common.hpp"
#include "fgl_kernels.hpp"
#include "fgl_split.hpp"

namespace fgl {

typedef float F32x16 __attribute__((ext_vector_type(16)));

// The rows that one step of a wave multiplies, as loaded (GROUPS row groups of the matrix instruction's depth).
template <typename T, int V>
struct WgradRows;

template <int V>
struct WgradRows<float, V> {
    static constexpr int kRows = 8;  // per step: four instructions of two rows
    typedef float Vec __attribute__((ext_vector_type(V), aligned(4)));
    Vec r[kRows / 2];
    // p: the step's first row (the same in all lanes); off: the lane's half-wave row and column
    static __device__ __forceinline__ uint32_t lane_offset(int col, int64_t ld, int half) { return (uint32_t)(half * ld) + (uint32_t)col; }
    __device__ __forceinline__ void load(const float* p, int64_t ld, uint32_t off)
    {
#pragma unroll
        for (int u = 0; u < kRows / 2; ++u) r[u] = *reinterpret_cast<const Vec*>(p + (int64_t)(2 * u) * ld + off);
    }
    // only the first n rows of the step exist
    __device__ __forceinline__ void load_tail(const float* p, int64_t ld, uint32_t off, int half, int n)
    {
#pragma unroll
        for (int u = 0; u < kRows / 2; ++u) {
            Vec z = {};
            r[u] = z;
            if (2 * u + half < n) r[u] = *reinterpret_cast<const Vec*>(p + (int64_t)(2 * u) * ld + off);
        }
    }
    __device__ __forceinline__ float at(int u, int c) const { return r[u][c]; }
    // sum[c] += column c of the lane's rows
    __device__ __forceinline__ void add_columns(float (&sum)[V]) const
    {
#pragma unroll
        for (int c = 0; c < V; ++c) sum[c] += (r[0][c] + r[1][c]) + (r[2][c] + r[3][c]);
    }
};

template <int V>
struct WgradRows<uint16_t, V> {
    static constexpr int kRows = 16;  // per step: one instruction of sixteen rows, eight per half-wave
    static constexpr int kWords = V == 4 ? 2 : 1;
    typedef uint32_t Vec2 __attribute__((ext_vector_type(2), aligned(4)));
    uint32_t r[8][kWords];
    __device__ __forceinline__ void load_one(const uint16_t* p, int i)
    {
        if constexpr (V == 1) {
            r[i][0] = *p;
        } else if constexpr (V == 2) {
            r[i][0] = *reinterpret_cast<const uint32_t*>(p);
        } else {
            const Vec2 v = *reinterpret_cast<const Vec2*>(p);
            r[i][0] = v[0];
            r[i][1] = v[1];
        }
    }
    static __device__ __forceinline__ uint32_t lane_offset(int col, int64_t ld, int half) { return (uint32_t)(8 * half * ld) + (uint32_t)col; }
    __device__ __forceinline__ void load(const uint16_t* p, int64_t ld, uint32_t off)
    {
#pragma unroll
        for (int i = 0; i < 8; ++i) load_one(p + (int64_t)i * ld + off, i);
    }
    __device__ __forceinline__ void load_tail(const uint16_t* p, int64_t ld, uint32_t off, int half, int n)
    {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
#pragma unroll
            for (int w = 0; w < kWords; ++w) r[i][w] = 0u;
            if (8 * half + i < n) load_one(p + (int64_t)i * ld + off, i);
        }
    }
    // column c of the lane's eight rows, as the instruction's operand
    __device__ __forceinline__ Bf16x8 column(int c) const { return bf16_column(r, c); }
    __device__ __forceinline__ void add_columns(float (&sum)[V]) const
    {
#pragma unroll
        for (int c = 0; c < V; ++c) {
            float s[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) s[i] = __uint_as_float((c & 1) ? r[i][c >> 1] & 0xFFFF0000u : r[i][c >> 1] << 16);
            sum[c] += ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
        }
    }
};

template <int VA, int VB>
__device__ __forceinline__ void wgrad_multiply(const WgradRows<float, VA>& a, const WgradRows<float, VB>& b, F32x16 (&acc)[VA * VB])
{
#pragma unroll
    for (int u = 0; u < WgradRows<float, VA>::kRows / 2; ++u)
#pragma unroll
        for (int i = 0; i < VA; ++i)
#pragma unroll
            for (int j = 0; j < VB; ++j)
                acc[i * VB + j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.at(u, i), b.at(u, j), acc[i * VB + j], 0, 0, 0);
}

template <int VA, int VB>
__device__ __forceinline__ void wgrad_multiply(const WgradRows<uint16_t, VA>& a, const WgradRows<uint16_t, VB>& b, F32x16 (&acc)[VA * VB])
{
    Bf16x8 fb[VB];
#pragma unroll
    for (int j = 0; j < VB; ++j) fb[j] = b.column(j);
#pragma unroll
    for (int i = 0; i < VA; ++i) {
        const Bf16x8 fa = a.column(i);
#pragma unroll
        for (int j = 0; j < VB; ++j) acc[i * VB + j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb[j], acc[i * VB + j], 0, 0, 0);
    }
}

// The rows of a step of the split form as loaded: eight per half-wave, V neighbouring columns a lane.
template <int V>
struct WgradEights {
    typedef float Vec __attribute__((ext_vector_type(V), aligned(4)));
    Vec r[8];
    static __device__ __forceinline__ uint32_t lane_offset(int col, int64_t ld, int half) { return (uint32_t)(8 * half * ld) + (uint32_t)col; }
    __device__ __forceinline__ void load(const float* p, int64_t ld, uint32_t off)
    {
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = *reinterpret_cast<const Vec*>(p + (int64_t)i * ld + off);
    }
    __device__ __forceinline__ void load_tail(const float* p, int64_t ld, uint32_t off, int half, int n)
    {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            Vec z = {};
            r[i] = z;
            if (8 * half + i < n) r[i] = *reinterpret_cast<const Vec*>(p + (int64_t)i * ld + off);
        }
    }
    // sign times column c in three parts, and the largest magnitude of it so far
    __device__ __forceinline__ void split(int c, float sign, SpU4 (&p)[3], uint32_t& rest, float& most) const
    {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = r[i][c] * sign;
        sp_split<true>(v, p, rest);
        sp_most(v, most);
    }
    __device__ __forceinline__ void add_columns(float (&sum)[V]) const
    {
#pragma unroll
        for (int c = 0; c < V; ++c) sum[c] += ((r[0][c] + r[1][c]) + (r[2][c] + r[3][c])) + ((r[4][c] + r[5][c]) + (r[6][c] + r[7][c]));
    }
};

struct WgradArgs {
    const void* a;
    const void* b;
    int64_t lda, ldb;
    int64_t k;
    int m, n;
    int tiles_n, tiles;   // tiles of C: along n, in all
    int splits;           // k splits, a multiple of eight where there is more than one tile
    int64_t k_per_split;  // rows of one split
    float* partial;       // [split][tile][register][lane]
    void* c;
    int64_t ldc;
    void* sum_a;          // (may be null) the column sums of A, m of them: a layer's bias gradient
    float* partial_sum;   // [split][tile along m][column]
};

// first column of lane i's vector (i in 0..31) in a tile
template <int V>
__device__ __forceinline__ int wgrad_column(int tile, int i, int n)
{
    const int c = (tile * 32 + i) * V;
    return c + V <= n ? c : n - V;
}

// acc += the products of the wave's rows between k0 and k1, and sum += the column sums of A's.  col_a, col_b: the lane's first
// column of either.
template <typename T, int VA, int VB>
__device__ __forceinline__ void wgrad_rows(const WgradArgs& g, int64_t k0, int64_t k1, int wave, int col_a, int col_b, bool sums, F32x16 (&acc)[VA * VB], float (&sum)[VA])
{
    const int half = lane_id() / 32;
    const T* pa = static_cast<const T*>(g.a);
    const T* pb = static_cast<const T*>(g.b);
    const uint32_t off_a = WgradRows<T, VA>::lane_offset(col_a, g.lda, half);
    const uint32_t off_b = WgradRows<T, VB>::lane_offset(col_b, g.ldb, half);
    // The wave's steps: rows k .. k + kRows - 1, then four steps (one per wave) further on; only the last may be short (or
    // empty).  The next step's rows are requested before the current ones are multiplied.  Nothing branches between the last
    // products and the first reads of the accumulators: a matrix instruction's results may be read a fixed number of
    // cycles later only, which the compiler (clang 22) was seen not to keep across such a branch.
    constexpr int kRows = WgradRows<T, VA>::kRows, kWaves = kBlock / kWave;
    constexpr int64_t kStep = (int64_t)kRows * kWaves;
    const int64_t first = k0 + (int64_t)wave * kRows;
    const int whole = k1 > first ? (int)((k1 - first - 1) / kStep) : 0;  // steps before the last one
    const T* ra = pa + first * g.lda;
    const T* rb = pb + first * g.ldb;
    WgradRows<T, VA> a0, a1;
    WgradRows<T, VB> b0, b1;
    if (whole > 0) {
        a0.load(ra, g.lda, off_a);
        b0.load(rb, g.ldb, off_b);
    } else {
        a0.load_tail(ra, g.lda, off_a, half, 0);  // (zeros)
        b0.load_tail(rb, g.ldb, off_b, half, 0);
    }
    for (int i = 1; i < whole; ++i) {
        ra += kStep * g.lda;
        rb += kStep * g.ldb;
        a1.load(ra, g.lda, off_a);
        b1.load(rb, g.ldb, off_b);
        if (sums) a0.add_columns(sum);
        __builtin_amdgcn_sched_barrier(0);  // (left alone, the compiler moves the loads behind the products to save registers)
        wgrad_multiply<VA, VB>(a0, b0, acc);
        a0 = a1;
        b0 = b1;
    }
    const int64_t last = first + whole * kStep;
    const int n = k1 - last < kRows ? (k1 > last ? (int)(k1 - last) : 0) : kRows;
    a1.load_tail(pa + last * g.lda, g.lda, off_a, half, n);
    b1.load_tail(pb + last * g.ldb, g.ldb, off_b, half, n);
    if (sums) {
        a0.add_columns(sum);
        a1.add_columns(sum);
    }
    wgrad_multiply<VA, VB>(a0, b0, acc);
    wgrad_multiply<VA, VB>(a1, b1, acc);
}

// The same in three bf16 parts a value, the wave's rows being others; true where the lane met values that have none (then acc is
// not the sum)
template <int VA, int VB>
__device__ __forceinline__ bool wgrad_split_rows(const WgradArgs& g, int64_t k0, int64_t k1, int wave, int col_a, int col_b, bool sums, F32x16 (&acc)[VA * VB],
                                                 float (&sum)[VA])
{
    constexpr int kRows = 16, kWaves = kBlock / kWave;
    constexpr int64_t kStep = (int64_t)kRows * kWaves;
    constexpr int kPa[6] = {2, 0, 1, 1, 0, 0}, kPb[6] = {0, 2, 1, 0, 1, 0};  // (the small products first)
    const int half = lane_id() / 32;
    const uint32_t off_a = WgradEights<VA>::lane_offset(col_a, g.lda, half);
    const uint32_t off_b = WgradEights<VB>::lane_offset(col_b, g.ldb, half);
    const int64_t first = k0 + (int64_t)wave * kRows;
    const int whole = k1 > first ? (int)((k1 - first - 1) / kStep) : 0;  // steps before the last one, which may be short or empty
    const float* ra = static_cast<const float*>(g.a) + first * g.lda;
    const float* rb = static_cast<const float*>(g.b) + first * g.ldb;
    const int64_t last = first + whole * kStep;
    const int n = k1 - last < kRows ? (k1 > last ? (int)(k1 - last) : 0) : kRows;
    WgradEights<VA> a;
    WgradEights<VB> b;
    uint32_t rest_a[VA], rest_b[VB];
    float most_a[VA], most_b[VB];
#pragma unroll
    for (int i = 0; i < VA; ++i) {
        rest_a[i] = 0;
        most_a[i] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < VB; ++j) {
        rest_b[j] = 0;
        most_b[j] = 0.0f;
    }
    auto load = [&](int i) {
        if (i < whole) {
            a.load(ra, g.lda, off_a);
            b.load(rb, g.ldb, off_b);
        } else {
            a.load_tail(ra, g.lda, off_a, half, n);
            b.load_tail(rb, g.ldb, off_b, half, n);
        }
        ra += kStep * g.lda;
        rb += kStep * g.ldb;
    };
    load(0);
    float sign = 1.0f;
    for (int s = 0; s <= whole; ++s) {
        if (sums) a.add_columns(sum);
        SpU4 pa[VA][3], pb[VB][3];
#pragma unroll
        for (int i = 0; i < VA; ++i) a.split(i, sign, pa[i], rest_a[i], most_a[i]);
#pragma unroll
        for (int j = 0; j < VB; ++j) b.split(j, 1.0f, pb[j], rest_b[j], most_b[j]);
        if (s < whole) load(s + 1);  // (on the way while these are multiplied)
        __builtin_amdgcn_sched_barrier(0);
        F32x16 part[VA * VB];
#pragma unroll
        for (int i = 0; i < VA; ++i)
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int j = 0; j < VB; ++j)
                    part[i * VB + j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(Bf16x8, pa[i][kPa[q]]), __builtin_bit_cast(Bf16x8, pb[j][kPb[q]]),
                                                                               q == 0 ? F32x16{} : part[i * VB + j], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < VA * VB; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[t][i] = fmaf(part[t][i], sign, acc[t][i]);
        sign = -sign;
    }
    bool odd = false;
#pragma unroll
    for (int t = 0; t < VA * VB; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) odd |= sp_odd(acc[t][i]);
    bool loses = false;
#pragma unroll
    for (int i = 0; i < VA; ++i) {
        rest_a[i] = (rest_a[i] | __shfl_xor(rest_a[i], 32, kWave)) & 0xFFFFu;
        loses |= rest_a[i] != 0;
    }
#pragma unroll
    for (int j = 0; j < VB; ++j) {
        rest_b[j] = (rest_b[j] | __shfl_xor(rest_b[j], 32, kWave)) & 0xFFFFu;
        loses |= rest_b[j] != 0;
    }
    if (__any(loses)) {
#pragma unroll
        for (int i = 0; i < VA; ++i) most_a[i] = fmaxf(most_a[i], __shfl_xor(most_a[i], 32, kWave));
#pragma unroll
        for (int j = 0; j < VB; ++j) most_b[j] = fmaxf(most_b[j], __shfl_xor(most_b[j], 32, kWave));
        const float terms = (float)(whole + 1) * kRows;
#pragma unroll
        for (int i = 0; i < VA; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 8 * (r / 4) + 4 * half + r % 4;  // of the tile: the lane with that column of A
                const bool row_loses = __shfl((int)rest_a[i], row, kWave) != 0;
                const float row_most = __shfl(most_a[i], row, kWave);
#pragma unroll
                for (int j = 0; j < VB; ++j)
                    odd |= !(fabsf(acc[i * VB + j][r]) >= sp_least(terms, row_loses, row_most, rest_b[j] != 0, most_b[j]));
            }
    }
    return odd;
}

template <typename T, int VA, int VB, bool SPLIT>
__global__ __launch_bounds__(kBlock, VA * VB >= 16 ? 1 : 2) void wgrad_kernel(const WgradArgs g)
{
    constexpr int kTiles = VA * VB;                    // 32x32 tiles of a wave
    constexpr int kChunk = kTiles < 4 ? kTiles : 4;    // of them added through LDS at a time
    constexpr int kWaves = kBlock / kWave;
    __shared__ float s_acc[kWaves][kChunk * 16][kWave];
    const int lane = lane_id();
    // The wave's number as a scalar: every branch around the matrix instructions below has to be a branch of the whole wave,
    // since they multiply in all lanes whatever the execution mask says.
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    // workgroup -> (split, tile): eight neighbouring splits (one per XCD) take turns, so the tiles of a split share an XCD
    const int group = (int)(blockIdx.x / (8u * (unsigned)g.tiles)), in_group = (int)(blockIdx.x % (8u * (unsigned)g.tiles));
    const int split = group * 8 + in_group % 8, tile = in_group / 8;
    if (split >= g.splits) return;  // (uniform over the workgroup)
    const int tm = tile / g.tiles_n, tn = tile % g.tiles_n;
    const int64_t k0 = (int64_t)split * g.k_per_split;
    const int64_t k1 = k0 + g.k_per_split < g.k ? k0 + g.k_per_split : g.k;
    const int col_a = wgrad_column<VA>(tm, lane % 32, g.m), col_b = wgrad_column<VB>(tn, lane % 32, g.n);
    F32x16 acc[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;
    // (the column sums of A ride on the workgroups of C's first column of tiles)
    const bool sums = g.sum_a != nullptr && tn == 0;
    float sum[VA];
#pragma unroll
    for (int i = 0; i < VA; ++i) sum[i] = 0.0f;

    if constexpr (SPLIT) {
        // (all waves of a workgroup or none; the sums of columns are right all the same)
        if (__syncthreads_or(wgrad_split_rows<VA, VB>(g, k0, k1, wave, col_a, col_b, sums, acc, sum))) {
            float unused[VA];
#pragma unroll
            for (int t = 0; t < kTiles; ++t) acc[t] = F32x16{};
            wgrad_rows<T, VA, VB>(g, k0, k1, wave, col_a, col_b, false, acc, unused);
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) {  // (read before the branch ends, see wgrad_rows)
                    float v = acc[t][i] + 0.0f;
                    asm volatile("" : "+v"(v));
                    acc[t][i] = v;
                }
        }
    } else {
        wgrad_rows<T, VA, VB>(g, k0, k1, wave, col_a, col_b, sums, acc, sum);
    }

    float* out = g.partial + ((int64_t)split * g.tiles + tile) * (kTiles * 16) * kWave;
#pragma unroll
    for (int q = 0; q < kTiles / kChunk; ++q) {
#pragma unroll
        for (int t = 0; t < kChunk; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) s_acc[wave][t * 16 + i][lane] = acc[q * kChunk + t][i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kChunk * 4; ++i) {  // each wave adds up a quarter of the registers
            const int r = wave * (kChunk * 4) + i;
            float s = s_acc[0][r][lane];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) s += s_acc[w][r][lane];
            out[(int64_t)(q * kChunk * 16 + r) * kWave + lane] = s;
        }
        __syncthreads();
    }
    if (!sums) return;
    float* s_sum = &s_acc[0][0][0];
#pragma unroll
    for (int i = 0; i < VA; ++i) {
        const float s = sum[i] + __shfl_xor(sum[i], 32, kWave);  // (the half-waves hold different rows of the same columns)
        if (lane < 32) s_sum[wave * (32 * VA) + lane * VA + i] = s;
    }
    __syncthreads();
    for (int i = (int)threadIdx.x; i < 32 * VA; i += kBlock) {
        float s = s_sum[i];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) s += s_sum[w * (32 * VA) + i];
        g.partial_sum[((int64_t)split * (g.tiles / g.tiles_n) + tm) * (32 * VA) + i] = s;
    }
}

// Adds the splits: a workgroup per (tile, accumulator register), four lanes of splits per output; behind those, a
// workgroup per 64 column sums of A.
template <typename T, int VA, int VB>
__global__ __launch_bounds__(kBlock) void wgrad_reduce_kernel(const WgradArgs g)
{
    constexpr int kTiles = VA * VB, kWaves = kBlock / kWave;
    __shared__ float s_sum[kWaves][kWave];
    const int lane = lane_id(), wave = (int)(threadIdx.x / kWave);
    const int tile = (int)(blockIdx.x / (kTiles * 16)), reg = (int)(blockIdx.x % (kTiles * 16));
    const bool sums = tile >= g.tiles;  // (uniform over the workgroup)
    const int sum_columns = g.tiles / g.tiles_n * 32 * VA;
    const int at = (int)(blockIdx.x - (unsigned)(g.tiles * kTiles * 16)) * kWave + lane;  // column sums only
    const int64_t stride = sums ? sum_columns : (int64_t)g.tiles * (kTiles * 16) * kWave;
    const float* p = sums ? g.partial_sum + (at < sum_columns ? at : 0) : g.partial + ((int64_t)tile * (kTiles * 16) + reg) * kWave + lane;
    float s = 0.0f;
    int q = wave;
    for (; q + 3 * kWaves < g.splits; q += 4 * kWaves) {
        const float v0 = p[q * stride], v1 = p[(q + kWaves) * stride], v2 = p[(q + 2 * kWaves) * stride], v3 = p[(q + 3 * kWaves) * stride];
        s += (v0 + v1) + (v2 + v3);
    }
    for (; q < g.splits; q += kWaves) s += p[q * stride];
    s_sum[wave][lane] = s;
    __syncthreads();
    if (wave != 0) return;
    s = (s_sum[0][lane] + s_sum[1][lane]) + (s_sum[2][lane] + s_sum[3][lane]);
    if (sums) {
        if (at >= sum_columns) return;
        const int col = wgrad_column<VA>(at / (32 * VA), at % (32 * VA) / VA, g.m) + at % VA;
        if constexpr (sizeof(T) == 4) static_cast<float*>(g.sum_a)[col] = s;
        else static_cast<__bf16*>(g.sum_a)[col] = (__bf16)s;
        return;
    }
    // accumulator register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of its 32x32 tile
    const int r = reg % 16, t = reg / 16;
    const int row = 8 * (r / 4) + 4 * (lane / 32) + r % 4;
    const int mm = wgrad_column<VA>(tile / g.tiles_n, row, g.m) + t / VB;
    const int nn = wgrad_column<VB>(tile % g.tiles_n, lane % 32, g.n) + t % VB;
    if constexpr (sizeof(T) == 4) static_cast<float*>(g.c)[(int64_t)mm * g.ldc + nn] = s;
    else static_cast<__bf16*>(g.c)[(int64_t)mm * g.ldc + nn] = (__bf16)s;
}

// Columns per lane along one side of C: what pads the least, the wider of two that pad alike.
static inline int wgrad_vec(int n, bool vectors, int widest)
{
    if (!vectors || n <= 32) return 1;
    int best = 1;
    int64_t pad = ceil_div(n, 32) * 32;
    for (int v = 2; v <= widest; v *= 2) {
        const int64_t p = ceil_div(n, 32 * v) * 32 * v;
        if (n >= v && p * 10 <= pad * 12) {  // (a fifth more columns is a fair price for a vector load twice as wide)
            best = v;
            if (p < pad) pad = p;
        }
    }
    return best;
}

struct WgradPlan {
    int va, vb;
    int tiles_n, tiles, splits;
    int64_t k_per_split;
    size_t sum_offset;  // of the column sums in the workspace
    size_t ws_bytes;
};

static WgradPlan wgrad_plan(int64_t k, int m, int n, bool va_ok, bool vb_ok, bool split)
{
    WgradPlan p;
    p.va = wgrad_vec(m, va_ok, split ? 2 : 4);
    p.vb = wgrad_vec(n, vb_ok, split ? 2 : 4);
    p.tiles_n = (int)ceil_div(n, 32 * p.vb);
    p.tiles = p.tiles_n * (int)ceil_div(m, 32 * p.va);
    // workgroups: one per CU with 16 tiles a wave (256 accumulators a lane), more of the smaller ones
    const int per_cu = p.va * p.vb >= 16 ? 1 : p.va * p.vb >= 8 || split ? 2 : 4;
    int64_t splits = 256 * per_cu / p.tiles;
    const int64_t most = ceil_div(k, 256);  // 256 rows and more per split: the sum over the splits costs as much as they do otherwise
    if (splits > most) splits = most;
    if (splits > 8) splits = splits / 8 * 8;
    // With many tiles eights of splits fill the chip badly (602 x 256 in 40 tiles: 320 workgroups of 512 places): the first
    // number of them that leaves less than an eighth of the places empty, also if it takes two rounds
    for (int64_t s = 8; split && splits < 32 && s <= 32 && s <= most; s += 8) {
        const int64_t rounds = ceil_div(s * p.tiles, 512) * 512;
        splits = s;
        if (s * p.tiles * 8 >= rounds * 7) break;
    }
    if (splits < 1) splits = 1;
    p.k_per_split = ceil_div(ceil_div(k, splits), 64) * 64;
    if (p.k_per_split < 64) p.k_per_split = 64;
    p.splits = (int)ceil_div(k, p.k_per_split);
    if (p.splits < 1) p.splits = 1;
    p.sum_offset = align_up((size_t)p.splits * p.tiles * p.va * p.vb * 16 * kWave * sizeof(float), 256);
    p.ws_bytes = p.sum_offset + align_up((size_t)p.splits * (p.tiles / p.tiles_n) * 32 * p.va * sizeof(float), 256);
    return p;
}

// Whether three parts a value pay: where the fp32 form has wide tiles, of which few waves hold 128 or 256 accumulators a lane
// (with narrow ones it is as fast or faster: us, fp32 / split, 64 x 64 k = 8000 11 / 12, 64 K 16 / 18; 96 x 40 k = 3000 9 / 11;
// 172 x 2 k = 20 K 11 / 12), and not where there is so much to multiply that reading the operands once for each tile of 64 is
// what counts (100 x 256 k = 107 K 68 / 65, 400 K 232 / 247; 256 x 256 k = 130 K 155 / 152, 200 K 227 / 237; with 65 to 128
// columns on one side, two tiles, 100 x 4000 k = 20 K 174 / 203, 100 x 602 k = 110 K 159 / 166, 100 x 1000 k = 60 K 142 / 136).
// A split's workgroups are one XCD's, so that fewer than eight splits leave XCDs idle; four times the tiles leave room for fewer
// of them where k allows few: k = 1000, 1000 x 1000 61 / 83 (four splits / two), 2000 x 602 104 / 162, 256 x 4000 61 / 82; k =
// 3000 119 / 79, 214 / 97, 120 / 77. Fewer rows than a step has are the fp32 form's, whose sums of one and two products are the
// more exact ones: rms errors against 64 bits, fp32 / split, k = 1 2.5e-8 / 3.5e-8, k = 2 3.1e-8 / 3.4e-8, k = 16 6.1e-8 /
// 3.4e-8, k = 17 6.5e-8 / 4.3e-8, k = 64 8.6e-8 / 5.5e-8.
static bool wgrad_split_pays(int64_t k, int m, int n)
{
    const int least = m < n ? m : n;
    if (k < 16 || wgrad_vec(m, true, 4) * wgrad_vec(n, true, 4) < 8 || (double)k * m * n > (least > 64 && least <= 128 ? 6e9 : 9e9)) return false;
    const int splits = wgrad_plan(k, m, n, true, true, true).splits;
    return splits >= 8 || splits >= wgrad_plan(k, m, n, true, true, false).splits;
}

static bool wgrad_vectors(int dtype, int cols, int64_t ld, const void* ptr)
{
    return dtype == FGL_F32 || (cols % 2 == 0 && ld % 2 == 0 && ((uintptr_t)ptr & 3) == 0);
}

template <typename T, int VA, int VB, bool SPLIT>
static int launch_wgrad(const WgradArgs& g, hipStream_t stream)
{
    const int64_t blocks = ceil_div(g.splits, 8) * 8 * g.tiles;
    hipLaunchKernelGGL((wgrad_kernel<T, VA, VB, SPLIT>), dim3((unsigned)blocks), dim3(kBlock), 0, stream, g);
    const int64_t sum_blocks = g.sum_a != nullptr ? ceil_div((int64_t)(g.tiles / g.tiles_n) * 32 * VA, kWave) : 0;
    hipLaunchKernelGGL((wgrad_reduce_kernel<T, VA, VB>), dim3((unsigned)(g.tiles * VA * VB * 16 + sum_blocks)), dim3(kBlock), 0, stream, g);
    FGL_CHECK_LAUNCH("wgrad_kernel");
    return FGL_OK;
}

template <typename T>
static int launch_wgrad_any(const WgradPlan& p, const WgradArgs& g, hipStream_t s)
{
#define FGL_WGRAD_CASE(A_, B_) if (p.va == A_ && p.vb == B_) return launch_wgrad<T, A_, B_, false>(g, s)
    FGL_WGRAD_CASE(4, 4);
    FGL_WGRAD_CASE(4, 2);
    FGL_WGRAD_CASE(4, 1);
    FGL_WGRAD_CASE(2, 4);
    FGL_WGRAD_CASE(2, 2);
    FGL_WGRAD_CASE(2, 1);
    FGL_WGRAD_CASE(1, 4);
    FGL_WGRAD_CASE(1, 2);
#undef FGL_WGRAD_CASE
    return launch_wgrad<T, 1, 1, false>(g, s);
}

}  // namespace fgl

using namespace fgl;

FGL_EXPORT size_t fgl_weight_grad_workspace_bytes_for(int64_t k, int m, int n, int dtype)
{
    if (k < 0 || m < 1 || n < 1) return 0;
    size_t most = 0;
    for (int i = 0; i < 4; ++i) {
        const size_t b = wgrad_plan(k, m, n, (i & 1) != 0, (i & 2) != 0, false).ws_bytes;
        if (b > most) most = b;
    }
    const size_t b = dtype == FGL_F32 && wgrad_split_pays(k, m, n) ? wgrad_plan(k, m, n, true, true, true).ws_bytes : 0;
    return b > most ? b : most;
}

FGL_EXPORT size_t fgl_weight_grad_workspace_bytes(int64_t k, int m, int n) { return fgl_weight_grad_workspace_bytes_for(k, m, n, FGL_F32); }

FGL_EXPORT int fgl_weight_grad(const void* d_a, int64_t lda, const void* d_b, int64_t ldb, int64_t k, int m, int n, int dtype,
                               void* d_c, int64_t ldc, void* d_sum_a, void* d_ws, size_t ws_bytes, void* stream)
{
    FGL_REQUIRE(k >= 0 && m >= 1 && n >= 1 && m <= 65536 && n <= 65536, "weight_grad: sizes %lld x %d x %d", (long long)k, m, n);
    FGL_REQUIRE(dtype == FGL_F32 || dtype == FGL_BF16, "weight_grad: unknown dtype %d", dtype);
    FGL_REQUIRE(lda >= m && ldb >= n && ldc >= n, "weight_grad: row stride smaller than the row length");
    FGL_REQUIRE(lda < (1 << 24) && ldb < (1 << 24), "weight_grad: row stride too large");  // (eight rows are spanned by 32-bit offsets)
    FGL_REQUIRE(d_c != nullptr && (k == 0 || (d_a && d_b)), "weight_grad: null pointer");
    const bool va = wgrad_vectors(dtype, m, lda, d_a), vb = wgrad_vectors(dtype, n, ldb, d_b);
    bool split = dtype == FGL_F32 && wgrad_split_pays(k, m, n);
    WgradPlan p = wgrad_plan(k, m, n, va, vb, split);
    if (split && ws_bytes < p.ws_bytes) {  // (a workspace for a longer k, which needs less where that is not in parts)
        split = false;
        p = wgrad_plan(k, m, n, va, vb, false);
    }
    if (d_ws == nullptr || ws_bytes < p.ws_bytes) {
        set_error("weight_grad: workspace too small (%zu < %zu)", ws_bytes, p.ws_bytes);
        return FGL_ERR_WORKSPACE;
    }
    WgradArgs g;
    g.a = d_a; g.b = d_b; g.lda = lda; g.ldb = ldb; g.k = k; g.m = m; g.n = n; g.tiles_n = p.tiles_n; g.tiles = p.tiles;
    g.splits = p.splits; g.k_per_split = p.k_per_split; g.partial = static_cast<float*>(d_ws); g.c = d_c; g.ldc = ldc;
    g.sum_a = d_sum_a; g.partial_sum = reinterpret_cast<float*>(static_cast<char*>(d_ws) + p.sum_offset);
    hipStream_t s = as_stream(stream);
    note_product(split ? "wgrad_kernel in parts" : "wgrad_kernel");
    if (split) return launch_wgrad<float, 2, 2, true>(g, s);  // (whoever is 128 wide in fours or 64 in twos is whole in twos)
    if (dtype == FGL_F32) return launch_wgrad_any<float>(p, g, s);
    return launch_wgrad_any<uint16_t>(p, g, s);
}
