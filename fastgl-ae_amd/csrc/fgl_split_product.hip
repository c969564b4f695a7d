// Products over the rows of a block in fp32 (what fgl_row_product.hip forms, which see), on the bf16 matrix cores: C[m, n] = A[m,
// k] B[k, n].
//
// (The parts: G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019; how they are summed and when they are not taken is this file's.)
//
// Why: the fp32 matrix instructions reach 157 TFLOP/s, the bf16 ones 2500.  An fp32 value is the sum of three bf16 values,
// exactly, so a product is six bf16 products and loses only terms below 2^-26 of it: a2 b0, a0 b2, a1 b1, a1 b0, a0 b1, a0 b0 of
// a = a0 + a1 + a2, b = b0 + b1 + b2, 2.6 times the rate.
//
// How exact.  Every product of two parts is exact, and what a matrix instruction adds up is cut to 26 bits of its largest term.
// So the 32 k of a chunk are added up from zero, the small products first, and only their sum is added to the accumulators, in
// fp32: errors of a sum of k terms grow with k / 32 where they grew with k.  Against 64-bit sums, 2-norm, normal / non-negative
// operands (the fp32 instructions in brackets): k = 100 5.8e-8 / 4.7e-8 (1.8e-7 / 1.4e-7), k = 256 7.0e-8 / 5.1e-8 (2.9e-7 /
// 2.5e-7), k = 800 1.1e-7 / 7.1e-8 (5.1e-7 / 3.8e-7).  Added to the accumulators directly the errors of k = 602 were those of the
// fp32 instructions and larger, because the cut then is at the accumulator's 26 bits.
// Values without such parts: infinite, not a
// number or rounded to infinity ones make results that are no finite numbers.  Values below 2^-110 may have bits below 2^-133,
// bf16's last, which are lost; they matter to a result that is not large beside them (sp_least), and subnormal results have no
// room for the small products. 32 columns of a tile with a result of these kinds are formed again in fp32 matrix instructions.
// (us, 107 K x 256 x 256, B transposed / not: 90 / 90; one column of B at 1e-36 191 / 232, where the fp32 kernel alone takes 161
// / 144; a hundredth of A's rows at 1e-37 158 / 181; a hundredth of A's values, or one row of B, at 1e-37, which change no
// result, 97 / 95.)
//
// What bounds it: for short k and few columns the pass over A and C, beyond that the matrix cores and the vector unit beside them.
//
// Split: a workgroup keeps its 32 NT columns of B in LDS, already in parts and in the order in which the lanes take them, and its
// waves go over the rows of A in tiles of 32, each by itself: no barrier after the first.  A lane reads its row of A straight to
// registers, a chunk ahead, and splits it; so the splitting costs each wave once for NT tiles, and no row is staged.  B is staged
// once for as many rows as there are, which is what a row tile a workgroup cannot do (both operands through LDS by tiles of 128 x
// 128: 107 K x 100 x 256 60 us where this takes 49). Beside each matrix instruction (32 cycles) the vector unit has room for
// about six others: the splitting of the next step (44 a step) and the addition of the last round's sums (16 a tile) are dealt
// out between them, which the compiler does not do by itself.  Left to its order, with the same instructions, 107 K x 256 x 256
// takes 96 us.
//
// Measured (MI355X, us: the fp32 instructions / the library / this; a transposed B costs no more here): 2.4 M x 100 x 64 550 / 511 /
// 345 (4.6 TB/s), 2.4 M x 64 x 100 449 / 625 / 332 (4.7 TB/s), 107 K x 100 x 256 78 / 81 / 51, 107 K x 256 x 256 149 / 138 / 90,
// 17 K x 256 x 256 42 / 25 / 27, 200 K x 128 x 128 85 / 81 / 50, 8192 x 602 x 256 27 / 27 / 26, 8192 x 256 x 602 42 / 36 / 28.
//
// Rows past the end repeat the last one and are not stored, nor are columns past the end, which repeat the last one too; the last
// step of k ends with k, and what the step before has of it is zero in LDS.  No access leaves the operands.
#include "fgl_common.hpp"
#include "fgl_kernels.hpp"
#include "fgl_row_product.hpp"
#include "fgl_split.hpp"

namespace fgl {

typedef float SpF4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kSpLds = 158 * 1024;  // of a CU, for B (the rest: the largest of each column)

// Eight values of a row of A, from its k number k0 on; only the first n of them exist.
__device__ __forceinline__ void sp_load(const float* p, float (&v)[8])
{
    const SpF4 a = *reinterpret_cast<const SpF4*>(p), b = *reinterpret_cast<const SpF4*>(p + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = a[j];
        v[4 + j] = b[j];
    }
}
__device__ __forceinline__ void sp_load_tail(const float* p, int n, float (&v)[8])
{
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        v[j] = 0.0f;
        if (j < n) v[j] = p[j];
    }
}

// Where step s starts: the last one ends with k (where k has 16 values at all), and B's image in LDS is zero for what the step before had.
__device__ __forceinline__ int sp_first(int s, int k)
{
    const int at = 16 * s;
    return k >= 16 && at + 16 > k ? k - 16 : at;
}


// The k of one product in steps of 16, two steps to a chunk.  (Where the steps are odd in number the last is one of zeros.)
__device__ __host__ __forceinline__ int sp_chunks(int k) { return (k + 31) / 32; }

// Column of tile t, lane i (of 32), from the workgroup's first one: a lane's columns are neighbours by ones, twos or fours (1 <<
// vl), as wide as its stores may be and no wider than they are aligned (n = 126 in misaligned vectors of four: 600 K x 64 x 126
// 164 us where 124 columns take 99).
__device__ __forceinline__ int sp_column(int vl, int t, int i) { return ((t >> vl) << (5 + vl)) + (i << vl) + (t & ((1 << vl) - 1)); }

// The steps of B's columns from col0 on -> img[step * NT + tile][part][lane], and the largest magnitude of each (magnitudes are
// in order as whole numbers too).  Four eights of k of one column a thread at a time, so that their loads are in flight together.
template <int NT, bool BT, int THREADS>
__device__ __forceinline__ void sp_stage(const RowProductSide& x, int steps, int col0, int n, int vl, SpU4* img, float* most, uint32_t* rest)
{
    constexpr int kCols = 32 * NT, kBatch = 4;
    const float* b = static_cast<const float*>(x.b);
    const int items = steps * 2 * kCols;
    for (int first = (int)threadIdx.x; first < items; first += THREADS * kBatch) {
        float v[kBatch][8];
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            const int at = first + i * THREADS < items ? first + i * THREADS : items - 1, oct = at / kCols;
            const int col = col0 + at % kCols < n ? col0 + at % kCols : n - 1;  // (columns past the end repeat the last one)
            const int own = 16 * (oct / 2) + oct % 2 * 8, k0 = sp_first(oct / 2, x.k) + oct % 2 * 8;
            const float* p = BT ? b + (int64_t)col * x.ldb + k0 : b + k0 * x.ldb + col;
            if (k0 == own && k0 + 8 <= x.k) {
                if constexpr (BT) {
                    sp_load(p, v[i]);
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[i][j] = p[j * x.ldb];
                }
            } else {  // the last step: what the step before has of it, and what lies past the end, is zero
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    v[i][j] = 0.0f;
                    if (k0 + j >= own - oct % 2 * 8 && k0 + j < x.k) v[i][j] = BT ? p[j] : p[j * x.ldb];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            const int at = first + i * THREADS, oct = at / kCols, col = at % kCols;
            if (at >= items) break;
            const int t = (col >> (5 + vl) << vl) + (col & ((1 << vl) - 1)), i_of = (col >> vl) & 31;
            float m = 0.0f;
            sp_most(v[i], m);
            atomicMax(reinterpret_cast<int*>(most + col), __float_as_int(m));
            SpU4 p[3];
            uint32_t r = 0;
            sp_split(v[i], p, r);
            if (sp_loses(r)) rest[col] = 1;
            SpU4* to = img + ((oct / 2) * NT + t) * 3 * kWave + oct % 2 * 32 + i_of;
#pragma unroll
            for (int q = 0; q < 3; ++q) to[q * kWave] = p[q];
        }
    }
}

// What a wave multiplies and what it has on the way.  A step of 16 k takes P = NT / 2 rounds of two tiles (one, where NT is 1); a
// round is six matrix instructions a tile, and the vector unit meanwhile adds the round before's sums to the accumulators and
// splits the step after's values of A.
template <int NT>
struct SpWave {
    static constexpr int kTiles = NT < 2 ? 1 : 2, kRounds = NT / kTiles;
    SpF32x16 acc[NT];
    SpF32x16 sum[2][kTiles];  // of this round and the one before
    SpU4 b[2][kTiles][3];     // B's values of this round and the next
    SpU4 a[2][3];             // A's of this step and the next
    float x[8], y[2][8];      // A's as loaded: the chunk's second step, the next chunk
    // of the row as far as it is split, and of the next chunk's first step: what tells whether bits are lost (sp_split), the
    // largest magnitude
    uint32_t rest, next_rest;
    float most, next_most;

    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = SpF32x16{};
        rest = 0;
        most = 0.0f;
    }
    template <int BUF>
    __device__ __forceinline__ void read_b(const SpU4* img)
    {
#pragma unroll
        for (int t = 0; t < kTiles; ++t)
#pragma unroll
            for (int p = 0; p < 3; ++p) b[BUF][t][p] = img[(t * 3 + p) * kWave];
    }
    // step U of a chunk; img: its B (of the lane), after: the next step's; r: the next step's values of A
    template <int U>
    __device__ __forceinline__ void step(const SpU4* img, const SpU4* after, const float (&r)[8])
    {
#pragma unroll
        for (int j = 0; j < kRounds; ++j) {
            constexpr int kPa[6] = {2, 0, 1, 1, 0, 0}, kPb[6] = {0, 2, 1, 0, 1, 0};
            const int buf = kRounds % 2 ? (U + j) & 1 : j & 1;
            const SpU4* ahead = j + 1 < kRounds ? img + (j + 1) * kTiles * 3 * kWave : after;
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int p = 0; p < 3; ++p) b[buf ^ 1][t][p] = ahead[(t * 3 + p) * kWave];
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int t = 0; t < kTiles; ++t)
                    sum[buf][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(Bf16x8, a[U & 1][kPa[q]]), __builtin_bit_cast(Bf16x8, b[buf][t][kPb[q]]),
                                                                          q == 0 ? SpF32x16{} : sum[buf][t], 0, 0, 0);
            const int before = (j + kRounds - 1) % kRounds * kTiles;
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[before + t][i] += sum[buf ^ 1][t][i];
            if (j == kRounds - 1) {
                sp_split(r, a[(U + 1) & 1], U == 0 ? rest : next_rest);
                sp_most(r, U == 0 ? most : next_most);
            }
#pragma unroll
            for (int i = 0; i < 6 * kTiles; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, kTiles == 1 ? 10 : kRounds == 1 ? 7 : 5, 0);
                if (i < 3 * kTiles) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // after the last step of a tile, which had ring position U
    template <int U>
    __device__ __forceinline__ void flush()
    {
        constexpr int kBuf = kRounds % 2 ? (U + kRounds - 1) & 1 : (kRounds - 1) & 1;
#pragma unroll
        for (int t = 0; t < kTiles; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[NT - kTiles + t][i] += sum[kBuf][t][i];
        sum[kBuf][0] = SpF32x16{};
        if constexpr (kTiles == 2) sum[kBuf][1] = SpF32x16{};
    }
};

// acc += one pair of operands, 32 columns, in fp32 matrix instructions.  a: the lane's row of A, col: its column of B.  Lanes of the lower
// half have the first four k of every eight, those of the upper half the others.
template <bool BT>
__device__ __forceinline__ void sp_plain(const float* a, const RowProductSide& x, int col, SpF32x16& acc)
{
    constexpr int U = 4;
    const int k = x.k, ldb = (int)x.ldb, half = lane_id() / 32;
    const float* b = static_cast<const float*>(x.b);
    const uint32_t off = BT ? 0 : (uint32_t)(U * half * ldb + col);  // (split_product_pays keeps ldb below 2^27)
    const float* bt = b + (int64_t)col * ldb;
    for (int k0 = 0; k0 < k; k0 += 2 * U) {
        const int kl = k0 + U * half;
        SpF4 va = {}, vb = {};
        if (kl + U <= k) {
            va = *reinterpret_cast<const SpF4*>(a + kl);
            if constexpr (BT) vb = *reinterpret_cast<const SpF4*>(bt + kl);
        } else {
#pragma unroll
            for (int j = 0; j < U; ++j) {
                if (kl + j < k) va[j] = a[kl + j];
                if (BT && kl + j < k) vb[j] = bt[kl + j];
            }
        }
        if constexpr (!BT) {
#pragma unroll
            for (int j = 0; j < U; ++j)
                if (kl + j < k) vb[j] = (b + (int64_t)(k0 + j) * ldb)[off];
        }
#pragma unroll
        for (int j = 0; j < U; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(va[j], vb[j], acc, 0, 0, 0);
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(0.0f, 0.0f, acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        float s = acc[i] + 0.0f;
        asm volatile("" : "+v"(s));
        acc[i] = s;
    }
}

// A tile of 32 rows to C, V neighbouring columns a lane.
template <int NT, int V, int FORM>
__device__ __forceinline__ void sp_store_tile(const RowProductArgs& g, int64_t row0, int col0, const SpF32x16 (&acc)[NT])
{
    int64_t ldc = g.ldc;
    int lane = lane_id();
    asm volatile("" : "+s"(ldc), "+v"(lane));  // (else what all widths make of them is kept in registers, and others spilled, all the while)
    const int half = lane / 32;
    float* out = static_cast<float*>(g.c) + (row0 + 4 * half) * ldc + col0;
    const bool rows = row0 + 32 <= g.m;  // (uniform)
#pragma unroll
    for (int q = 0; q < NT / V; ++q) {
        const int at = 32 * V * q + lane % 32 * V, left = g.n - col0 - at;
        float add[V];
#pragma unroll
        for (int t = 0; t < V; ++t) {
            add[t] = 0.0f;
            if (g.bias != nullptr && t < left) add[t] = static_cast<const float*>(g.bias)[col0 + at + t];
        }
        // What C holds is read for several rows at a time: the compiler keeps each row's loads behind the stores before them, and
        // a row a round trip made 895 K x 64 x 47 added to C 266 us, this 126 (600 K x 64 x 128, in vectors, 177 and 158).
        constexpr int kBatch = FORM == kRpAdd ? 16 / V : 16;
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += kBatch) {
            typedef float Vec __attribute__((ext_vector_type(V), aligned(4)));
            float* p[kBatch];
            Vec held[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int r = r0 + i, row = 8 * (r / 4) + r % 4;
                p[i] = out + at + row * ldc;
                held[i] = Vec{};
                if constexpr (FORM == kRpAdd) {
                    if (rows && left >= V) {
                        held[i] = *reinterpret_cast<const Vec*>(p[i]);
                    } else {
#pragma unroll
                        for (int t = 0; t < V; ++t)
                            if (row0 + 4 * half + row < g.m && t < left) held[i][t] = p[i][t];
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int r = r0 + i, row = 8 * (r / 4) + r % 4;
                float v[V];
#pragma unroll
                for (int t = 0; t < V; ++t) {
                    v[t] = acc[q * V + t][r] + add[t];
                    if constexpr (FORM == kRpAdd) v[t] += held[i][t];
                }
                if (rows && left >= V) {
                    rp_store<float, V>(p[i], v);
                } else {
#pragma unroll
                    for (int t = 0; t < V; ++t)
                        if (row0 + 4 * half + row < g.m && t < left) p[i][t] = v[t];
                }
            }
        }
    }
}

template <int NT, int W, bool BT, int FORM>
__global__ __launch_bounds__(W * kWave, 2) void split_product_kernel(const RowProductArgs g)
{
    constexpr int kThreads = W * kWave;
    extern __shared__ SpU4 s_img[];
    __shared__ float s_most[2][32 * NT];     // of each column: its largest magnitude, and whether its values lose bits
    __shared__ uint32_t s_rest[2][32 * NT];
    const int lane = lane_id(), half = lane / 32;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const unsigned per_group = 8u * (unsigned)g.tiles_n;
    const int64_t rb = (int64_t)(blockIdx.x / per_group) * 8 + blockIdx.x % per_group % 8;
    const int col0 = (int)(blockIdx.x % per_group / 8) * 32 * NT;
    if (rb * W * 32 >= g.m) return;  // (uniform over the workgroup: no row tile for it)
    const int chunks0 = sp_chunks(g.side[0].k), chunks = chunks0 + (FORM == kRpSum ? sp_chunks(g.side[1].k) : 0);
    const int64_t row_tiles = (g.m + 31) / 32, stride = g.row_blocks * W;
    int64_t tile = rb * W + wave;

    // the lane's row of a tile, from its half-wave's first k on
    auto row_of = [&](const RowProductSide& x, int64_t t) {
        int64_t row = t * 32 + lane % 32;
        if (row >= g.m) row = g.m - 1;
        return static_cast<const float*>(x.a) + row * x.lda + half * 8;
    };
    // what is loaded next: chunk `at` of tile `ahead`, whose rows begin at p0 and p1
    int64_t ahead = tile;
    int at = 0;
    const float* p0 = row_of(g.side[0], ahead);
    const float* p1 = FORM == kRpSum ? row_of(g.side[1], ahead) : nullptr;
    auto load = [&](float (&r)[2][8]) {
        const bool second = FORM == kRpSum && at >= chunks0;
        const float* p = second ? p1 : p0;
        const int k = second ? g.side[1].k : g.side[0].k, first = 32 * (second ? at - chunks0 : at);
        if (k >= 16) {
            sp_load(p + (first < k - 16 ? first : k - 16), r[0]);
            sp_load(p + (first + 16 < k - 16 ? first + 16 : k - 16), r[1]);
        } else {
            sp_load_tail(p, k - half * 8, r[0]);
            sp_load_tail(p, 0, r[1]);
        }
        if (++at == chunks) {
            at = 0;
            if (ahead + stride < row_tiles) ahead += stride;
            p0 = row_of(g.side[0], ahead);
            if constexpr (FORM == kRpSum) p1 = row_of(g.side[1], ahead);
        }
    };
    SpWave<NT> w;
    load(w.y);
    if (threadIdx.x < 64 * NT) {  // (64 NT <= kThreads)
        (&s_most[0][0])[threadIdx.x] = 0.0f;
        (&s_rest[0][0])[threadIdx.x] = 0;
    }
    __syncthreads();
    sp_stage<NT, BT, kThreads>(g.side[0], 2 * chunks0, col0, g.n, g.vec_log, s_img, s_most[0], s_rest[0]);
    if constexpr (FORM == kRpSum) sp_stage<NT, BT, kThreads>(g.side[1], 2 * (chunks - chunks0), col0, g.n, g.vec_log, s_img + chunks0 * 2 * NT * 3 * kWave, s_most[1], s_rest[1]);
    __syncthreads();
    if (tile >= row_tiles) return;  // (uniform over the wave; no barrier follows)
    bool columns_lose = false;
    for (int i = lane; i < 64 * NT; i += kWave) columns_lose |= (&s_rest[0][0])[i] != 0;
    columns_lose = __any(columns_lose);
    w.clear();
#pragma unroll
    for (int t = 0; t < SpWave<NT>::kTiles; ++t) w.sum[1][t] = SpF32x16{};
    w.next_rest = 0;
    sp_split(w.y[0], w.a[0], w.next_rest);
    w.next_most = 0.0f;
    sp_most(w.y[0], w.next_most);
#pragma unroll
    for (int j = 0; j < 8; ++j) w.x[j] = w.y[1][j];
    const SpU4* img = s_img + lane;
    w.template read_b<0>(img);
    for (;;) {
        for (int c = 0; c < chunks; ++c) {
            load(w.y);
            w.rest |= w.next_rest;
            w.next_rest = 0;
            w.most = w.most < w.next_most ? w.next_most : w.most;
            w.next_most = 0.0f;
            const SpU4* after = c + 1 == chunks ? s_img + lane : img + 2 * NT * 3 * kWave;
            __builtin_amdgcn_sched_barrier(0);
            w.template step<0>(img, img + NT * 3 * kWave, w.x);
            w.template step<1>(img + NT * 3 * kWave, after, w.y[0]);
            img = after;
#pragma unroll
            for (int j = 0; j < 8; ++j) w.x[j] = w.y[1][j];
        }
        w.template flush<1>();
        SpF32x16 (&acc)[NT] = w.acc;
        const int64_t row0 = tile * 32;
        uint32_t odd = 0;  // bit t: tile t has a sum that is not to be had in parts
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) odd |= sp_odd(acc[t][i]) ? 1u << t : 0u;
        const bool row_loses = sp_loses(w.rest | __shfl_xor(w.rest, 32, kWave));
        if (columns_lose || __any(row_loses || odd != 0)) {  // (uniform)
            int own = lane % 32;
            asm volatile("" : "+v"(own));  // (else the compiler keeps what follows from it in registers all the while)
            auto row_again = [&](const RowProductSide& x) {
                const int64_t row = tile * 32 + own < g.m ? tile * 32 + own : g.m - 1;
                return static_cast<const float*>(x.a) + row * x.lda;
            };
            // (sums of fewer than 1024 terms, which is more than B's room allows; the larger of two pairs' values for either)
            float row_most[16];  // of the rows of the lane's sums: negative where the row loses bits
            const float mine = fmaxf(w.most, __shfl_xor(w.most, 32, kWave));
#pragma unroll
            for (int i = 0; i < 16; ++i) row_most[i] = __shfl(row_loses ? -mine : mine, 8 * (i / 4) + 4 * half + i % 4, kWave);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int c = sp_column(g.vec_log, t, own), col = col0 + c < g.n ? col0 + c : g.n - 1;
                const bool column_loses = (s_rest[0][c] | s_rest[1][c]) != 0;
                const float column_most = fmaxf(s_most[0][c], s_most[1][c]);
                bool small = (odd >> t & 1) != 0;
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    small |= !(fabsf(acc[t][i]) >= sp_least(1024.0f, row_most[i] < 0.0f, fabsf(row_most[i]), column_loses, column_most));
                if (!__any(small)) continue;
                acc[t] = SpF32x16{};
                sp_plain<BT>(row_again(g.side[0]), g.side[0], col, acc[t]);
                if constexpr (FORM == kRpSum) sp_plain<BT>(row_again(g.side[1]), g.side[1], col, acc[t]);
            }
            w.template read_b<0>(s_img + lane);  // (what was read ahead: its registers are free above)
        }
        if (NT >= 4 && g.vec_log == 2) sp_store_tile<NT, NT < 4 ? 1 : 4, FORM>(g, row0, col0, acc);
        else if (NT >= 2 && g.vec_log == 1) sp_store_tile<NT, NT < 2 ? 1 : 2, FORM>(g, row0, col0, acc);
        else sp_store_tile<NT, 1, FORM>(g, row0, col0, acc);
        tile += stride;
        if (tile >= row_tiles) return;
        w.clear();
    }
}

static size_t sp_lds(const RowProductArgs& g, int nt) { return (size_t)(sp_chunks(g.side[0].k) + sp_chunks(g.side[1].k)) * 2 * nt * 3 * kWave * sizeof(SpU4); }

// Row blocks, 8 at a time, one to an XCD with all of its tiles along n.  An XCD has `places` for workgroups at once, one or two a CU,
// and one more than that begins when the others end: 7 tiles of 128 columns in 64 places are 9 row blocks (63), not 10.  Where much would
// be left empty (13 tiles: 4 row blocks, 52) more of them in up to four rounds may end sooner: a workgroup takes as long as its waves have
// row tiles, and two tiles' time to stage B; six tenths of that in a last round that has the CUs to itself, so that half rounds count too.
// (us, with one block more than fits / with this: 209 K x 64 x 896 248 / 209, 100 K x 128 x 376 95 / 77, added to C 168 / 112, 119 K x (256 +
// 256) x 165 302 / 210, 80 K x 256 x 1064 424 / 302; whole rounds only / with this: 19 K x 128 x 2970 126 / 113.)
static int64_t sp_row_blocks(int64_t row_tiles, int waves, int per_cu, int64_t tiles_n)
{
    const int64_t places = 32 * per_cu, want = ceil_div(ceil_div(row_tiles, waves), 8);  // (of an XCD: a tile a wave)
    int64_t best = 1, least = INT64_MAX;
    for (int64_t halves = 2; halves <= 8; ++halves) {
        int64_t n = places * halves / (2 * tiles_n);
        if (n < 1) n = 1;
        if (n > want) n = want;
        const int64_t rest = n * tiles_n % places, last = rest == 0 ? 0 : per_cu == 2 && rest <= 32 && n * tiles_n > places ? 6 : 10;
        const int64_t time = (n * tiles_n / places * 10 + last) * (2 + ceil_div(row_tiles, 8 * n * waves));
        if (time < least) {
            least = time;
            best = n;
        }
    }
    return best * 8;
}

template <int NT, int W, bool BT, int FORM>
static int launch_split_product(RowProductArgs g, hipStream_t stream)
{
    const size_t lds = sp_lds(g, NT);
    g.tiles_n = (int)ceil_div(g.n, 32 * NT);
    // eight waves a CU (two a SIMD, as the registers allow), in as many workgroups as their LDS allows
    int64_t per_cu = kSpLds / (int64_t)lds;
    if (per_cu > 8 / W) per_cu = 8 / W;
    // as many neighbouring columns a lane as every row's start allows
    const uint64_t starts = (uintptr_t)g.c | (uint64_t)g.ldc * sizeof(float);
    g.vec_log = NT >= 4 && starts % 16 == 0 ? 2 : NT >= 2 && starts % 8 == 0 ? 1 : 0;
    g.row_blocks = sp_row_blocks(ceil_div(g.m, 32), W, (int)per_cu, g.tiles_n);
    const int64_t blocks = ceil_div(g.row_blocks, 8) * 8 * g.tiles_n;
    FGL_REQUIRE(blocks <= 0x7FFFFFFF, "row_product: grid too large");
    hipLaunchKernelGGL((split_product_kernel<NT, W, BT, FORM>), dim3((unsigned)blocks), dim3(W * kWave), lds, stream, g);
    FGL_CHECK_LAUNCH("split_product_kernel");
    return FGL_OK;
}

// Columns of a workgroup: 64, so that a split value of A serves two tiles and B fits up to k = 416; 32 for fewer columns or a
// longer k; 128 where k is short and the pass over A is what counts (2.4 M x 64 x 100: 325 us against 404; 200 K x 128 x 128,
// with one workgroup of four waves left a CU, 50 against 46).
static int sp_tiles(const RowProductArgs& g)
{
    const int steps = 2 * (sp_chunks(g.side[0].k) + sp_chunks(g.side[1].k));
    if (g.n > 64 && steps <= 4) return 4;
    return g.n > 32 && sp_lds(g, 2) <= (size_t)kSpLds ? 2 : 1;
}

// Whether the split pays, against the fp32 instructions' kernel, which has nothing to stage first and pads less.  A step here is
// 32 k and 32 to 128 columns: the line lies at 1.6e8 multiplications, higher by what k and the columns are padded (us, that kernel /
// this: 909 K x 8 x 33 42 / 70, 106 K x 33 x 66 19 / 22, but 140 K x 33 x 100 28 / 24), by the staging of a longer k (200 x 128: 13 K
// rows 12 / 15, 20 K 21 / 15; 602 x 64: 7800 13 / 22, 13 K 26 / 23), and where fewer than 1100 tiles of 32 rows leave more than half of
// the chip's 2048 places for waves empty (100 + 100 x 64: 29 K 13 / 17).  Of 900 products of 17 to 832 k, 2 to
// 3000 columns and 8e7 to 1.2e9 multiplications it took 0.8 % longer than the faster one, and 10 more than a tenth longer than that
// kernel (22 x 85 added to C, 265 K rows, 41 / 58; the others up to 1.18).
// Up to 32 k, of which half a chunk or more may be zeros, the line lies twice as far out and the pass over C is what counts: this is
// ahead where that kernel goes over A three times (130 M results: 18 x 92 222 / 138, 12 x 92 209 / 149; 30 M: 18 x 91 33 / 40), in
// narrow tiles (25 M and 130 M: 18 x 33 48 / 45, 256 / 249, 18 x 64 32 / 24, 158 / 126; but 16 x 33 36 / 45, 202 / 253, 18 x 16 46 / 57)
// and, of 17 k and more, where a row is one workgroup's or whole lines of 128 bytes are (18 x 100 145 / 135, 18 x 128 128 / 119, 18 x
// 256 123 / 108, 27 x 256, 38 M, 48 / 30; but 16 x 128, 240 M, 200 / 212, 24 x 127 137 / 245, 24 x 254 147 / 192, 24 x 380 141 / 166).
// One to three terms are that kernel's, which rounds their sum more exactly.  Odd rows in tiles of 128 columns, stored value by value,
// need a k that hides that (130 M: 40 x 127 194 / 260, 40 x 126 195 / 213, 40 x 380 202 / 176; 64 x 125, 75 M, 150 / 142).
// Workgroups of one row block go to one XCD, eight blocks at a time, so that fewer than 2000 rows leave XCDs idle: 1000 x 256 x
// 4000 22 / 36, 500 x 602 x 16000 192 / 356, 250 x 832 x 30000 521 / 909, 2000 x 256 x 4000 44 / 39.  Results as few as 1.6e6 take
// that many rows' worth twice: 3000 x 602 x 602 30 / 38, 4000 x 400 x 400 21 / 22.
bool split_product_pays(const RowProductArgs& g)
{
    const int k = g.side[0].k + g.side[1].k;
    if (sp_lds(g, 1) > (size_t)kSpLds || g.m < 2000 || (g.side[0].ldb | g.side[1].ldb) >> 27 != 0) return false;
    const double outputs = (double)g.m * g.n;
    if (outputs < (g.m < 5000 ? 2.1e6 : 1.6e6)) return false;
    const int tiles = sp_tiles(g);
    const int64_t padded_k = 32 * (sp_chunks(g.side[0].k) + sp_chunks(g.side[1].k)), column_tiles = ceil_div(g.n, 32 * tiles);
    const uint64_t starts = (uintptr_t)g.c | (uint64_t)g.ldc * sizeof(float);
    if (k < 4 || (k <= 16 && (g.n <= 64 || g.n > 96))) return false;
    if (k <= 32 && (g.n <= 32 || (g.n > 96 && starts % (column_tiles == 1 ? 16 : 128) != 0))) return false;
    if (k < 56 && g.n > 96 && tiles == 4 && starts % 8 != 0) return false;
    double line = 1.6e8 + 1e6 * (double)(padded_k > 128 ? padded_k - 128 : 0);
    line *= (double)padded_k / k * (double)(column_tiles * tiles) / (double)ceil_div(g.n, 32);
    if (ceil_div(g.m, 32) * column_tiles < 1100) line *= 1.3;
    if (k <= 32) line *= 2.0;
    return outputs * k >= line;
}

template <bool BT, int FORM>
static int launch_split_product_any(const RowProductArgs& g, hipStream_t stream)
{
    const int nt = sp_tiles(g);
    const bool one_a_cu = sp_lds(g, nt) * 2 > (size_t)kSpLds;  // then of eight waves, otherwise two of four
    if (nt == 4) return launch_split_product<4, 4, BT, FORM>(g, stream);
    if (nt == 2) return one_a_cu ? launch_split_product<2, 8, BT, FORM>(g, stream) : launch_split_product<2, 4, BT, FORM>(g, stream);
    return one_a_cu ? launch_split_product<1, 8, BT, FORM>(g, stream) : launch_split_product<1, 4, BT, FORM>(g, stream);
}

int split_product(const RowProductArgs& g, bool b_transposed, int form, hipStream_t stream)
{
    if (form == kRpSum) return b_transposed ? launch_split_product_any<true, kRpSum>(g, stream) : launch_split_product_any<false, kRpSum>(g, stream);
    if (form == kRpAdd) return b_transposed ? launch_split_product_any<true, kRpAdd>(g, stream) : launch_split_product_any<false, kRpAdd>(g, stream);
    return b_transposed ? launch_split_product_any<true, kRpOne>(g, stream) : launch_split_product_any<false, kRpOne>(g, stream);
}

}  // namespace fgl
