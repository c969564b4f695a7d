// A dense layer's product over the rows of a block: C[m, n] = sum over k of A[m, k] * B[k, n] (+ bias[n]), with m the node count of
// a block -- 10^2 .. 10^6, another one with every mini-batch -- and k, n layer widths.  B is the layer's weight, either [k, n] or,
// transposed, [n, k] (the reference forms these products with torch::mm, cuda_operators/aggregate_acc.cpp:144,188,371,402).
//
// Why not the library: it looks for a kernel by the exact sizes on every call, and a new m each time means 60-80 us of host time
// per product (74 against 12 through here), which is what a training step over mini-batches waited for: GCN step 1000 -> 840 us, GAT 1270 ->
// 890..940, GraphSAGE in bf16 1430..1630 -> 1110..1140 (three runs; the autograd thread makes two of them uneven).  Where such products
// gain is ops._forms_row_product's rule.
//
// What bounds it: in fp32 the matrix cores, in bf16 the one pass over A and C.  Large fp32 products go to fgl_split_product.hip, which forms them on the bf16
// matrix cores; the line is split_product_pays.
//
// Tile: a wave holds (32 VA) x (32 VB) outputs in its accumulators.  Nothing goes through LDS: the order of the k within a step
// is free, so lane i of a half-wave reads its own row of A with one 16-byte load along k (half 0 the step's first values, half 1 the rest) and
// has the operands of four matrix instructions (fp32; in bf16 of one, v_mfma_f32_32x32x16_bf16 wants eight consecutive k per lane).
// B comes the same way where it is transposed, and with one VB-wide load per k where it is not.  A lane's VB columns are
// neighbours, so C is stored in whole vectors, 32 lanes side by side.  B is read by every wave; it is a few hundred
// kilobytes that stay in the L2s, and the waves of a workgroup read it at the same time through one L1.
// Workgroups that share rows of A (different columns of C) are neighbours on one XCD.
// The next step's operands are requested before the current ones are multiplied.
//
// Measured (MI355X, us, the library's kernel / this one, the same sizes again and again): fp32 107 K x 100 x 256 81 / 78, 107 K x 256 x 256
// 138 / 144 (97 TFLOP/s), 200 K x 128 x 128 81 / 85; bf16 107 K x 100 x 256 29 / 24, 107 K x 256 x 256 29 / 39; a transposed B, whose loads touch a
// line per lane, costs up to an eighth more in fp32 and, from k = 128 on, a third in bf16 (107 K x 256 x 256: 27 / 52).
//
// Rows past the end repeat the last one and are not stored; a lane whose columns would leave the row takes the row's last VB columns
// (bit-equal copies of its neighbour's); k past the end is zero in both operands.  No access leaves the operands.
#include "fgl_common.hpp"
#include "fgl_kernels.hpp"
#include "fgl_row_product.hpp"

namespace fgl {

typedef float RpF32x16 __attribute__((ext_vector_type(16)));
typedef float RpF4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t RpU4 __attribute__((ext_vector_type(4), aligned(4)));

// One lane's values of a step: kLane values along k of one row (A, or a column of a transposed B).
template <typename T>
struct RpRow;
template <>
struct RpRow<float> {
    static constexpr int kLane = 4;  // per half-wave: a step is 8 k
    RpF4 v;
    __device__ __forceinline__ void load(const float* p) { v = *reinterpret_cast<const RpF4*>(p); }
    __device__ __forceinline__ void load_tail(const float* p, int n)
    {
#pragma unroll
        for (int j = 0; j < kLane; ++j) {
            v[j] = 0.0f;
            if (j < n) v[j] = p[j];
        }
    }
};
template <>
struct RpRow<uint16_t> {
    static constexpr int kLane = 8;  // per half-wave: a step is 16 k
    RpU4 v;
    __device__ __forceinline__ void load(const uint16_t* p) { v = *reinterpret_cast<const RpU4*>(p); }
    __device__ __forceinline__ void load_tail(const uint16_t* p, int n)
    {
#pragma unroll
        for (int j = 0; j < kLane / 2; ++j) {
            uint32_t lo = 0, hi = 0;
            if (2 * j < n) lo = p[2 * j];
            if (2 * j + 1 < n) hi = p[2 * j + 1];
            v[j] = lo | hi << 16;
        }
    }
    __device__ __forceinline__ Bf16x8 operand() const { return __builtin_bit_cast(Bf16x8, v); }
};

// One lane's values of a step of an untransposed B: kLane rows (k) of VB neighbouring columns.
template <typename T, int VB>
struct RpCols;
template <int VB>
struct RpCols<float, VB> {
    typedef float Vec __attribute__((ext_vector_type(VB), aligned(4)));
    Vec r[4];
    __device__ __forceinline__ void load_one(const float* p, int j) { r[j] = *reinterpret_cast<const Vec*>(p); }
    __device__ __forceinline__ void zero(int j) { r[j] = Vec{}; }
};
template <int VB>
struct RpCols<uint16_t, VB> {
    static constexpr int kWords = VB == 4 ? 2 : 1;
    typedef uint32_t Vec2 __attribute__((ext_vector_type(2), aligned(4)));
    uint32_t r[8][kWords];
    __device__ __forceinline__ void load_one(const uint16_t* p, int j)
    {
        if constexpr (VB == 1) {
            r[j][0] = *p;
        } else if constexpr (VB == 2) {
            r[j][0] = *reinterpret_cast<const uint32_t*>(p);
        } else {
            const Vec2 v = *reinterpret_cast<const Vec2*>(p);
            r[j][0] = v[0];
            r[j][1] = v[1];
        }
    }
    __device__ __forceinline__ void zero(int j)
    {
#pragma unroll
        for (int w = 0; w < kWords; ++w) r[j][w] = 0u;
    }
    // column c of the lane's eight rows, as the instruction's operand
    __device__ __forceinline__ Bf16x8 operand(int c) const { return bf16_column(r, c); }
};

template <typename T, int VA, int VB, bool BT>
struct RpStep {
    static constexpr int kLane = RpRow<T>::kLane;
    RpRow<T> a[VA];
    RpRow<T> bt[BT ? VB : 1];
    RpCols<T, VB> bn;  // (unused where B is transposed, and then no registers)

    // k0: the half-wave's first k of the step; a whole step
    __device__ __forceinline__ void load(const T* const (&pa)[VA], const T* pb, int64_t ldb, int k0)
    {
#pragma unroll
        for (int i = 0; i < VA; ++i) a[i].load(pa[i] + k0);
        if constexpr (BT) {
#pragma unroll
            for (int t = 0; t < VB; ++t) bt[t].load(pb + t * ldb + k0);
        } else {
#pragma unroll
            for (int j = 0; j < kLane; ++j) bn.load_one(pb + (int64_t)(k0 + j) * ldb, j);
        }
    }
    // only the first n of the half-wave's values exist (n may be <= 0)
    __device__ __forceinline__ void load_tail(const T* const (&pa)[VA], const T* pb, int64_t ldb, int k0, int n)
    {
#pragma unroll
        for (int i = 0; i < VA; ++i) a[i].load_tail(pa[i] + k0, n);
        if constexpr (BT) {
#pragma unroll
            for (int t = 0; t < VB; ++t) bt[t].load_tail(pb + t * ldb + k0, n);
        } else {
#pragma unroll
            for (int j = 0; j < kLane; ++j) {
                bn.zero(j);
                if (j < n) bn.load_one(pb + (int64_t)(k0 + j) * ldb, j);
            }
        }
    }
    __device__ __forceinline__ void multiply(RpF32x16 (&acc)[VA * VB]) const
    {
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int j = 0; j < kLane; ++j)
#pragma unroll
                for (int i = 0; i < VA; ++i)
#pragma unroll
                    for (int t = 0; t < VB; ++t) {
                        float b;
                        if constexpr (BT) b = bt[t].v[j];
                        else b = bn.r[j][t];
                        acc[i * VB + t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i].v[j], b, acc[i * VB + t], 0, 0, 0);
                    }
        } else {
#pragma unroll
            for (int t = 0; t < VB; ++t) {
                Bf16x8 b;
                if constexpr (BT) b = bt[t].operand();
                else b = bn.operand(t);
#pragma unroll
                for (int i = 0; i < VA; ++i) acc[i * VB + t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i].operand(), b, acc[i * VB + t], 0, 0, 0);
            }
        }
    }
};

// acc += the products of one pair of operands.  row0: the wave's first row; col: the lane's first column.
template <typename T, int VA, int VB, bool BT>
__device__ __forceinline__ void rp_side(const RowProductSide& side, int64_t row0, int64_t m, int col, RpF32x16 (&acc)[VA * VB])
{
    constexpr int kLane = RpRow<T>::kLane, kStep = 2 * kLane;
    const int lane = lane_id(), half = lane / 32, k = side.k;
    const T* pa[VA];
#pragma unroll
    for (int i = 0; i < VA; ++i) {
        const int64_t row = row0 + 32 * i + lane % 32;
        pa[i] = static_cast<const T*>(side.a) + (row < m ? row : m - 1) * side.lda;
    }
    const T* pb = static_cast<const T*>(side.b) + (BT ? (int64_t)col * side.ldb : (int64_t)col);
    // Steps before the last one are whole.  As in wgrad_kernel nothing branches between the last products and the first reads of
    // the accumulators, and every branch around a product is one of the whole wave.
    const int whole = (k - 1) / kStep;
    RpStep<T, VA, VB, BT> cur, next;
    int k0 = half * kLane;
    if (whole > 0) cur.load(pa, pb, side.ldb, k0);
    else cur.load_tail(pa, pb, side.ldb, k0, 0);  // (zeros)
    for (int s = 1; s < whole; ++s) {
        k0 += kStep;
        next.load(pa, pb, side.ldb, k0);
        __builtin_amdgcn_sched_barrier(0);  // (left alone, the compiler moves the loads behind the products to save registers)
        cur.multiply(acc);
        cur = next;
    }
    k0 = whole * kStep + half * kLane;
    if (k % kStep == 0) next.load(pa, pb, side.ldb, k0);
    else next.load_tail(pa, pb, side.ldb, k0, k - k0);
    cur.multiply(acc);
    next.multiply(acc);
}

template <typename T, int VA, int VB, bool BT, int FORM>
__global__ __launch_bounds__(kBlock, VA * VB >= 4 ? 2 : 4) void row_product_kernel(const RowProductArgs g)
{
    const int lane = lane_id();
    const int half = lane / 32;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    // workgroup -> (rows, columns): eight neighbouring row groups (one per XCD) take turns, so the tiles of a row group share an XCD
    const unsigned per_group = 8u * (unsigned)g.tiles_n;
    const int64_t rb = (int64_t)(blockIdx.x / per_group) * 8 + blockIdx.x % per_group % 8;
    const int tn = (int)(blockIdx.x % per_group / 8);
    const int64_t row0 = (rb * (kBlock / kWave) + wave) * (32 * VA);
    if (rb >= g.row_blocks || row0 >= g.m) return;  // (uniform over the wave)

    int col = (tn * 32 + lane % 32) * VB;
    const bool past_end = FORM == kRpAdd && col >= g.n;  // (adds nothing: the columns that it repeats are another lane's)
    if (col + VB > g.n) col = g.n - VB;
    RpF32x16 acc[VA * VB];
#pragma unroll
    for (int t = 0; t < VA * VB; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;
    float add[VB];
#pragma unroll
    for (int t = 0; t < VB; ++t) {
        add[t] = 0.0f;
        if (g.bias != nullptr) {
            if constexpr (sizeof(T) == 4) add[t] = static_cast<const float*>(g.bias)[col + t];
            else add[t] = __uint_as_float((uint32_t)static_cast<const uint16_t*>(g.bias)[col + t] << 16);
        }
    }

    rp_side<T, VA, VB, BT>(g.side[0], row0, g.m, col, acc);
    constexpr bool kKeep = FORM == kRpSum && sizeof(T) == 2;
    uint32_t kept[kKeep ? VA * VB : 1][8];  // the first product's values, two to a word
    if constexpr (FORM == kRpSum) {
        if constexpr (kKeep) {
#pragma unroll
            for (int t = 0; t < VA * VB; ++t)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    uint32_t w = rp_bf16_bits(acc[t][2 * i]) | rp_bf16_bits(acc[t][2 * i + 1]) << 16;
                    asm volatile("" : "+v"(w));
                    kept[t][i] = w;
                }
#pragma unroll
            for (int t = 0; t < VA * VB; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;
        }
        rp_side<T, VA, VB, BT>(g.side[1], row0, g.m, col, acc);
    }

    // Every sum leaves the accumulators here, before the branches around the stores: the empty statement keeps the compiler from moving
    // the additions behind them, which it did.  (fp32 107 K x 256 x 256: 149 us with them behind, 144 here; other sizes alike.)
#pragma unroll
    for (int i = 0; i < VA; ++i)
#pragma unroll
        for (int t = 0; t < VB; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float s = acc[i * VB + t][r] + add[t];
                if constexpr (FORM != kRpOne && sizeof(T) == 2) s = __uint_as_float(rp_bf16_bits(s) << 16);
                if constexpr (kKeep) s += __uint_as_float(r & 1 ? kept[i * VB + t][r / 2] & 0xFFFF0000u : kept[i * VB + t][r / 2] << 16);
                asm volatile("" : "+v"(s));
                acc[i * VB + t][r] = s;
            }

    // accumulator register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32 of its 32x32 tile
#pragma unroll
    for (int i = 0; i < VA; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t row = row0 + 32 * i + 8 * (r / 4) + 4 * half + r % 4;
            float v[VB];
#pragma unroll
            for (int t = 0; t < VB; ++t) v[t] = acc[i * VB + t][r];
            if (row < g.m && !past_end) {
                T* p = static_cast<T*>(g.c) + row * g.ldc + col;
                if constexpr (FORM == kRpAdd) rp_add<T, VB>(p, v);
                rp_store<T, VB>(p, v);
            }
        }
}

template <typename T, int VA, int VB, bool BT, int FORM>
static int launch_row_product(RowProductArgs g, hipStream_t stream)
{
    g.tiles_n = (int)ceil_div(g.n, 32 * VB);
    g.row_blocks = ceil_div(g.m, (int64_t)(kBlock / kWave) * 32 * VA);
    const int64_t blocks = ceil_div(g.row_blocks, 8) * 8 * g.tiles_n;
    FGL_REQUIRE(blocks <= 0x7FFFFFFF, "row_product: grid too large");
    hipLaunchKernelGGL((row_product_kernel<T, VA, VB, BT, FORM>), dim3((unsigned)blocks), dim3(kBlock), 0, stream, g);
    FGL_CHECK_LAUNCH("row_product_kernel");
    return FGL_OK;
}

// Tile: what pads n least, wide tiles where they still make a thousand waves (four per CU).  The last vector of a row is moved back to end with
// it and repeats columns of its neighbour, which for 129 columns in twos, or 514 in fours, is another workgroup's: harmless where both store
// the same values, but a sum would be added twice, so sums go to C in vectors only if a row is a whole number of them.
template <typename T, bool BT, int FORM>
static int launch_row_product_any(const RowProductArgs& g, bool vectors, hipStream_t stream)
{
    const int64_t pad1 = ceil_div(g.n, 32) * 32;
    int vb = 1;
    for (int v = 2; v <= 4 && vectors; v *= 2) {
        const int64_t p = ceil_div(g.n, 32 * v) * 32 * v;
        const int64_t waves = ceil_div(g.m, 32) * (p / (32 * v));
        if (g.n >= v && p * 10 <= pad1 * 12 && waves >= 1024 && (FORM != kRpAdd || g.n % v == 0)) vb = v;
    }
    // A bf16 sum keeps the first product's values besides the accumulators: no tall tiles.  An fp32 one goes on in the same accumulators; it gains by
    // tall tiles where there is enough to multiply (us, tiles of 32 / 64 rows: 87 K rows of 2 x 256 x 256 276 / 242, 2 x 100 x 256 128 / 115, 200 K of 2 x 256 x 64
    // 235 / 200, 2 x 128 x 128 192 / 180; but 2 x 100 x 100 146 / 150, 2 x 64 x 64 51 / 53, 2 x 50 x 47 45 / 49).
    constexpr bool kTall = FORM != kRpSum || sizeof(T) == 4;
    const bool tall = kTall && vb >= 2 && ceil_div(g.m, 64) * ceil_div(g.n, 32 * vb) >= 2048 &&
                      (FORM != kRpSum || (int64_t)(g.side[0].k + g.side[1].k) * g.n >= 32768);
    if constexpr (kTall) {
        if (vb == 4 && tall) return launch_row_product<T, 2, 4, BT, FORM>(g, stream);
        if (vb == 2 && tall) return launch_row_product<T, 2, 2, BT, FORM>(g, stream);
    }
    if (vb == 4) return launch_row_product<T, 1, 4, BT, FORM>(g, stream);
    if (vb == 2) return launch_row_product<T, 1, 2, BT, FORM>(g, stream);
    return launch_row_product<T, 1, 1, BT, FORM>(g, stream);
}

}  // namespace fgl

using namespace fgl;

static thread_local const char* g_product = "";
void fgl::note_product(const char* kernel) { g_product = kernel; }
FGL_EXPORT const char* fgl_product_last_kernel(void) { return g_product; }

template <int FORM>
static int row_product(const RowProductSide& one, const RowProductSide& two, int b_transposed, int64_t m, int n, int dtype, const void* d_bias,
                       void* d_c, int64_t ldc, void* stream)
{
    FGL_REQUIRE(dtype == FGL_F32 || dtype == FGL_BF16, "row_product: unknown dtype %d", dtype);
    FGL_REQUIRE(m >= 0 && n >= 1 && n <= 65536 && ldc >= n, "row_product: %lld rows of %d columns, %lld apart", (long long)m, n, (long long)ldc);
    RowProductArgs g;
    memset(&g, 0, sizeof(g));
    g.side[0] = one; g.side[1] = two; g.bias = d_bias; g.c = d_c; g.ldc = ldc; g.m = m; g.n = n;
    bool vectors = true;
    for (int i = 0; i < (FORM == kRpSum ? 2 : 1); ++i) {
        const RowProductSide& x = g.side[i];
        FGL_REQUIRE(x.k >= 1 && x.k <= 65536, "row_product: sizes %lld x %d x %d", (long long)m, x.k, n);
        FGL_REQUIRE(x.lda >= x.k && x.ldb >= (b_transposed ? x.k : n), "row_product: row stride smaller than the row length");
        if (m == 0) continue;
        FGL_REQUIRE(x.a && x.b && d_c, "row_product: null pointer");
        if (dtype == FGL_F32) continue;
        // bf16 moves in words: every row that is read along k starts on one, and so does every vector of C (and of an untransposed B)
        FGL_REQUIRE(x.lda % 2 == 0 && (uintptr_t)x.a % 4 == 0 && (!b_transposed || (x.ldb % 2 == 0 && (uintptr_t)x.b % 4 == 0)),
                    "row_product: bf16 rows must start on 4-byte boundaries");
        vectors = vectors && n % 2 == 0 && ldc % 2 == 0 && (uintptr_t)d_c % 4 == 0 && (b_transposed || (x.ldb % 2 == 0 && (uintptr_t)x.b % 4 == 0));
    }
    if (m == 0) return FGL_OK;
    hipStream_t s = as_stream(stream);
    const bool split = dtype == FGL_F32 && split_product_pays(g);
    note_product(split ? "split_product_kernel" : "row_product_kernel");
    if (split) return split_product(g, b_transposed != 0, FORM, s);
    if (dtype == FGL_F32) return b_transposed ? launch_row_product_any<float, true, FORM>(g, true, s) : launch_row_product_any<float, false, FORM>(g, true, s);
    return b_transposed ? launch_row_product_any<uint16_t, true, FORM>(g, vectors, s) : launch_row_product_any<uint16_t, false, FORM>(g, vectors, s);
}

FGL_EXPORT int fgl_row_product(const void* d_a, int64_t lda, const void* d_b, int64_t ldb, int b_transposed, int64_t m, int k, int n, int dtype,
                               const void* d_bias, void* d_c, int64_t ldc, void* stream)
{
    return row_product<kRpOne>(RowProductSide{d_a, d_b, lda, ldb, k}, RowProductSide{nullptr, nullptr, 0, 0, 0}, b_transposed, m, n, dtype, d_bias, d_c,
                               ldc, stream);
}

FGL_EXPORT int fgl_row_product_sum(const void* d_a0, int64_t lda0, const void* d_b0, int64_t ldb0, int k0, const void* d_a1, int64_t lda1,
                                   const void* d_b1, int64_t ldb1, int k1, int b_transposed, int64_t m, int n, int dtype, const void* d_bias,
                                   void* d_c, int64_t ldc, void* stream)
{
    return row_product<kRpSum>(RowProductSide{d_a0, d_b0, lda0, ldb0, k0}, RowProductSide{d_a1, d_b1, lda1, ldb1, k1}, b_transposed, m, n, dtype, d_bias,
                               d_c, ldc, stream);
}

FGL_EXPORT int fgl_row_product_add(const void* d_a, int64_t lda, const void* d_b, int64_t ldb, int b_transposed, int64_t m, int k, int n, int dtype,
                                   void* d_c, int64_t ldc, void* stream)
{
    return row_product<kRpAdd>(RowProductSide{d_a, d_b, lda, ldb, k}, RowProductSide{nullptr, nullptr, 0, 0, 0}, b_transposed, m, n, dtype, nullptr, d_c,
                               ldc, stream);
}
