// ar_split.hpp -- exact three-term bf16 splits of fp32 values, for products at
// fp32 accuracy on the bf16 matrix cores (ar_gemm_f32.hip, ar_attn_f32.hip).
//
//   x = hi + mid + lo,  hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid
// (8 significant bits each: 24 in all, and both differences are exact), and
//   x y = lo hi + hi lo + mid mid + mid hi + hi mid + hi hi
// with the dropped terms below 2^-25 of the product.
#pragma once

#include "ar_common.hpp"

namespace ar {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// The split of values e, e + 1 of an item of 8.  The two exact differences are
// dot products of the rounded pair with (-1, 0) / (0, -1): one
// v_dot2_f32_bf16 where a widening and a subtraction would be two, 3.5 VALU
// per value instead of 5.5.  The constants go through scalar registers: as an
// inline constant -1.0 the hardware reads the fp32 pattern, whose low half is
// zero.
__device__ __forceinline__ void split2(float x0, float x1, int e, bf16x8& hi, bf16x8& mid, bf16x8& lo) {
    unsigned c0 = 0x0000BF80u, c1 = 0xBF800000u;
    asm("" : "+s"(c0), "+s"(c1));
    const bf16x2 s0 = __builtin_bit_cast(bf16x2, c0), s1 = __builtin_bit_cast(bf16x2, c1);
    bf16x2 h, m;
    h[0] = (bf16)x0;
    h[1] = (bf16)x1;
    const float r0 = __builtin_amdgcn_fdot2_f32_bf16(h, s0, x0, false);
    const float r1 = __builtin_amdgcn_fdot2_f32_bf16(h, s1, x1, false);
    m[0] = (bf16)r0;
    m[1] = (bf16)r1;
    hi[e] = h[0];
    hi[e + 1] = h[1];
    mid[e] = m[0];
    mid[e + 1] = m[1];
    lo[e] = (bf16)__builtin_amdgcn_fdot2_f32_bf16(m, s0, r0, false);
    lo[e + 1] = (bf16)__builtin_amdgcn_fdot2_f32_bf16(m, s1, r1, false);
}

// 16-byte unit slot of a K-major LDS tile of U units per row: the 16 rows one
// phase of a fragment read touches (one unit each) fill all 64 banks once.
template <int U>
__device__ __forceinline__ int kslot(int r, int c) {
    static_assert(U == 4 || U == 8 || U == 16, "32-, 64- or 128-deep tiles");
    return U == 4   ? r * 4 + (c ^ ((r >> 2) & 3))
           : U == 8 ? r * 8 + (c ^ ((r >> 1) & 7))
                    : r * 16 + (c ^ (r & 15));
}

}  // namespace ar
