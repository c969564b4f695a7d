// fp32 values as sums of three bf16 values, for products on the bf16 matrix cores (fgl_split_product.hip says what that is worth and how exact it is).
#pragma once

#include "fgl_common.hpp"

namespace fgl {

typedef float SpF32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t SpU4 __attribute__((ext_vector_type(4)));

// Eight fp32 values as three bf16 operands: v = p[0] + p[1] + p[2] to the last bit (while v's last bit is no smaller than bf16's, 2^-133).  (v_dot2 with
// (-1, 0) and (0, -1) would take a part off in one instruction instead of two, but does not run beside a matrix instruction: one a MFMA takes 34 cycles to 45.)
__device__ __forceinline__ void sp_split(const float (&v)[8], SpU4 (&p)[3])
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
            if (s == 2) break;
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
// Whether a row or a column whose largest magnitude is m may lose bits to bf16's range: its values are off by 2^-134 at most, 2^-49 of anything from here on.
__device__ __forceinline__ bool sp_small(float m) { return m > 0.0f && m < 0x1p-85f; }

}  // namespace fgl
