// fp32 products on the bf16 matrix cores of gfx950, at fp32 accuracy.
//
// A float is the sum of three bf16 values, exactly: the upper 8 bits of its significand (cut off), the next 8 (rounded
// to nearest) and what is left, which fits 8 more.  Of the nine products of two such sums six are formed; the three left
// out (mid*lo, lo*mid, lo*lo) are below 2^-22 of a product and of either sign.  Products of bf16 values are exact in the
// matrix core and are added up in fp32.
// Why: v_mfma_f32_32x32x2_f32 does 32 multiply-adds a cycle and SIMD unit, v_mfma_f32_32x32x16_bf16 512, so for 16384 six
// passes of it take 192 cycles where the fp32 ones take 512, and the split costs about 6 vector instructions an element,
// which run beside the bf16 matrix core.
// An infinity has no such sum (inf - inf), so a tile whose result is not finite throughout is computed again with fp32
// instructions by the kernels that use this: NaN and infinities come out as they always did.  Parts below the smallest
// bf16 number are lost: operands keep full precision down to 2^-109 (1e-33).
#pragma once

#include <hip/hip_runtime.h>

typedef __bf16 fc_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 fc_bf16x2 __attribute__((ext_vector_type(2)));
typedef float fc_floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t fc_uintx4 __attribute__((ext_vector_type(4)));

// Two floats to their three parts, packed in pairs.
__device__ __forceinline__ void fc_split2(float a, float b, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
    hi = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
    fc_floatx2 r = {a - __builtin_bit_cast(float, ua & 0xffff0000u), b - __builtin_bit_cast(float, ub & 0xffff0000u)};
    mid = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, fc_bf16x2));
    fc_floatx2 q = {r[0] - __builtin_bit_cast(float, mid << 16), r[1] - __builtin_bit_cast(float, mid & 0xffff0000u)};
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(q, fc_bf16x2));
}

// Eight values of one row or column, consecutive in the reduction, to the operand words of the three parts; the parts
// lie `plane` 16-byte words apart.
__device__ __forceinline__ void fc_split8(const float (&v)[8], fc_uintx4 *dst, int plane) {
    fc_uintx4 h, m, l;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t a, b, c;
        fc_split2(v[2 * i], v[2 * i + 1], a, b, c);
        h[i] = a; m[i] = b; l[i] = c;
    }
    dst[0] = h;
    dst[plane] = m;
    dst[2 * plane] = l;
}

// LDS image of one 16-deep stage of both operands, in 16-byte words: [part][depth / 8][row] of A, then the same of B
// with columns.  Lane l of a 32x32x16 product holds row l % 32, depths 8 * (l / 32) .. + 7: one word, neighbouring lanes
// neighbouring words, no bank conflicts.
template <int BM, int BN>
struct fc_split_stage {
    static constexpr int A_PLANE = 2 * BM, B_PLANE = 2 * BN, WORDS = 3 * (A_PLANE + B_PLANE);
};

// acc += A * B over one stage, smallest products first.  `as`, `bs`: this lane's word of the first part and 32-wide block.
template <int MI, int NI, int A_PLANE, int B_PLANE, class Acc>
__device__ __forceinline__ void fc_split_products(const fc_uintx4 *as, const fc_uintx4 *bs, Acc (&acc)[MI][NI]) {
    fc_bf16x8 a[3][MI], b[3][NI];
#pragma unroll
    for (int q = 2; q >= 0; q--) {
#pragma unroll
        for (int mi = 0; mi < MI; mi++) a[q][mi] = __builtin_bit_cast(fc_bf16x8, as[q * A_PLANE + mi * 32]);
#pragma unroll
        for (int ni = 0; ni < NI; ni++) b[2 - q][ni] = __builtin_bit_cast(fc_bf16x8, bs[(2 - q) * B_PLANE + ni * 32]);
    }
    constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
    for (int q = 0; q < 6; q++)
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
                acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[q]][mi], b[pb[q]][ni], acc[mi][ni], 0, 0, 0);
}

// Whether any of a lane's accumulators is an infinity or a NaN.
template <int MI, int NI, class Acc>
__device__ __forceinline__ bool fc_not_finite(const Acc (&acc)[MI][NI]) {
    float z = 0.f;
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int i = 0; i < 16; i++) z = __builtin_fmaf(acc[mi][ni][i], 0.f, z);
    return z != z;
}
