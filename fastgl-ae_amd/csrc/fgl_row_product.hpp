// What the kernels of a dense layer's product over rows share: operands, and how a lane's columns of a row are stored.
#pragma once

#include "fgl_common.hpp"

namespace fgl {

struct RowProductSide {
    const void* a;
    const void* b;
    int64_t lda, ldb;
    int k;  // 0: no such pair
};
struct RowProductArgs {
    RowProductSide side[2];  // C = A0 B0 + A1 B1
    const void* bias;
    void* c;
    int64_t ldc, m;
    int n;
    int tiles_n;          // tiles of C along n
    int64_t row_blocks;   // workgroups along m
    int vec_log;          // (split products) log2 of the neighbouring columns a lane stores
};

__device__ __forceinline__ uint32_t rp_bf16_bits(float v) { return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v); }

// v += what p holds
template <typename T, int VB>
__device__ __forceinline__ void rp_add(const T* p, float (&v)[VB])
{
    if constexpr (sizeof(T) == 4) {
        typedef float Vec __attribute__((ext_vector_type(VB), aligned(4)));
        const Vec o = *reinterpret_cast<const Vec*>(p);
#pragma unroll
        for (int t = 0; t < VB; ++t) v[t] += o[t];
    } else if constexpr (VB == 1) {
        v[0] += __uint_as_float((uint32_t)*p << 16);
    } else {
        typedef uint32_t Vec __attribute__((ext_vector_type(VB / 2), aligned(4)));
        const Vec o = *reinterpret_cast<const Vec*>(p);
#pragma unroll
        for (int t = 0; t < VB; ++t) v[t] += __uint_as_float(t & 1 ? o[t / 2] & 0xFFFF0000u : o[t / 2] << 16);
    }
}

template <typename T, int VB>
__device__ __forceinline__ void rp_store(T* p, const float (&v)[VB])
{
    if constexpr (sizeof(T) == 4) {
        typedef float Vec __attribute__((ext_vector_type(VB), aligned(4)));
        Vec o;
#pragma unroll
        for (int t = 0; t < VB; ++t) o[t] = v[t];
        *reinterpret_cast<Vec*>(p) = o;
    } else if constexpr (VB == 1) {
        *reinterpret_cast<__bf16*>(p) = (__bf16)v[0];
    } else {
        typedef __bf16 Vec __attribute__((ext_vector_type(VB), aligned(4)));
        Vec o;
#pragma unroll
        for (int t = 0; t < VB; ++t) o[t] = (__bf16)v[t];
        *reinterpret_cast<Vec*>(p) = o;
    }
}

// FORM: one product (kRpOne), two of them and their sum (kRpSum: a layer's own rows with one weight and its gathered rows with another, in one
// pass over C where the products and their sum were five), or a product added to what C holds (kRpAdd).  In bf16 a product is rounded to
// bf16 before it is added to another or to C, as it would be if it were stored in between.
constexpr int kRpOne = 0, kRpSum = 1, kRpAdd = 2;

// fp32 products on the bf16 matrix cores: whether they pay for these sizes, and one of them
bool split_product_pays(const RowProductArgs& g);
int split_product(const RowProductArgs& g, bool b_transposed, int form, hipStream_t stream);

}  // namespace fgl
