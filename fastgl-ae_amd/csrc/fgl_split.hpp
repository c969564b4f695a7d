// fp32 values as sums of three bf16 values, for products on the bf16 matrix cores (fgl_split_product.hip says what that is worth
// and how exact it is).
#pragma once

#include "fgl_common.hpp"

namespace fgl {

typedef float SpF32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t SpU4 __attribute__((ext_vector_type(4)));

// Eight fp32 values as three bf16 operands: v = p[0] + p[1] + p[2] to the last bit, while v's last bit is no smaller than bf16's,
// 2^-133.  What the third part has to hold goes to `rest`: a bf16 value's low half is zero, so rest has bits there (sp_loses) if
// and only if one of the values loses some; each of them is off by 2^-134 at most.  (v_dot2 with (-1, 0) and (0, -1) would take a
// part off in one instruction instead of two, but does not run beside a matrix instruction: one a MFMA takes 34 cycles to 45.)
// PINNED: by an instruction that the compiler does not move; otherwise it takes all of the weight gradient's splitting behind the
// loads of the next rows and between the matrix instructions there (100 x 256, k = 107 K: 68.4 us, 65 so; the products over rows,
// which say themselves what goes where, 60.2 / 61.5).
template <bool PINNED = false>
__device__ __forceinline__ void sp_split(const float (&v)[8], SpU4 (&p)[3], uint32_t& rest)
{
    typedef __bf16 B2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float x = v[2 * j], y = v[2 * j + 1];
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            B2 h;
            h[0] = (__bf16)x;
            h[1] = (__bf16)y;
            uint32_t w = __builtin_bit_cast(uint32_t, h);
            p[s][j] = w;
            if (s == 2) {
                if constexpr (PINNED) asm("v_or3_b32 %0, %1, %2, %0" : "+v"(rest) : "v"(x), "v"(y));
                else rest |= __float_as_uint(x) | __float_as_uint(y);
                break;
            }
            x -= __uint_as_float(w << 16);
            y -= __uint_as_float(w & 0xFFFF0000u);
        }
    }
}

// m = the largest magnitude of m and eight values (what is not a number is passed over)
__device__ __forceinline__ void sp_most(const float (&v)[8], float& m)
{
#pragma unroll
    for (int j = 0; j < 8; j += 2) asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(v[j]), "v"(v[j + 1]));
}
// (Telling exactly which rows and columns lose bits costs as many instructions as their largest values do, 2 of the 63 us of that
// weight gradient.  Judged by a largest value below 2^-85 alone, tiny values beside large ones lost bits unseen, and columns that
// lose nothing were formed twice.)
__device__ __forceinline__ bool sp_loses(uint32_t rest) { return (rest & 0xFFFFu) != 0; }
// What a sum of n products has to reach for the values that lose bits, on either side or both, to be 2^-26 of it together: n 2^-134
// times the largest value that they are multiplied with.
__device__ __forceinline__ float sp_least(float n, bool a_loses, float a_most, bool b_loses, float b_most)
{
    return n * 0x1p-108f * ((a_loses ? b_most : 0.0f) + (b_loses ? a_most : 0.0f));
}
// Whether a sum is not to be had in parts: infinite, not a number, or so small that the parts' products have no room for their bits
__device__ __forceinline__ bool sp_odd(float sum) { return __builtin_amdgcn_classf(sum, 0x297); }

}  // namespace fgl
