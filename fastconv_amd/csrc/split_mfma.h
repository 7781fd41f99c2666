// fp32 products on the bf16 matrix cores of gfx950, at fp32 accuracy.
//
// A float is the sum of three bf16 values, exactly: the float rounded to bf16 (8 significant bits), what that leaves
// rounded again, and what is left then, which is a whole number of the float's last places and fits 8 bits.  (Three-part
// bf16 operands with the smallest partial products left out: Henry, Tang and Heinecke, "Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations", 2019.)
// Of the nine products of two such sums six are formed; the three left out (mid*lo, lo*mid, lo*lo) are together below
// 2^-24 of a product, the most that one fp32 multiply-add rounds off, and of either sign.  Products of bf16 values are
// exact in the matrix core and are added up in fp32, but each of its additions rounds off up to a last place of the sum:
// the five small products have sums of their own, added to those of hi*hi at the end, so that they round at their own size.
// Error against 64 bits over that of v_mfma_f32_32x32x2_f32, measured over sums of 256 normal terms of which n are not
// zero: 1.03 for n = 1, 0.67 for 4, 0.46 for 16, 0.38 for 64, 0.31 for 256.  (All six in one sum: 1.37, 1.82, 1.87, 1.47,
// 0.82, and 10 % less time with 128x128 tiles, 2 % with 64x64 ones; the first part cut off instead of rounded: 1.64 for n = 1.)
// Why: v_mfma_f32_32x32x2_f32 does 32 multiply-adds a cycle and SIMD unit, v_mfma_f32_32x32x16_bf16 512, so for 16384 six
// passes of it take 192 cycles where the fp32 ones take 512, and the split costs about 7 vector instructions an element,
// which run beside the bf16 matrix core.
// Operands are multiplied by 2^24 first and sums by 2^-48 last: the parts of the smallest subnormal float are then normal
// bf16 numbers, and the split is exact over the whole lower range (without it parts below 2^-133 are lost, 2^-10 of an
// operand of 2^-124).  One multiplication an element, 1 to 3 % of a launch.
// An infinity has no such sum (inf - inf), and scaled operands from 2^104 and sums from 2^80 on overflow.  Values that are
// not finite are formed again with fp32 instructions by the kernels that use this, the others keep what they are: NaN,
// infinities and large values come out as they always did, and a value depends on its own row and column alone.  A tile
// with such a value runs through its reduction a second time: 256 -> 256 channels at 56x56, batch 32, one NaN 178 -> 194 us,
// one in every tile 441 us (all on fp32 instructions: 225).
#pragma once

#include <hip/hip_runtime.h>

typedef __bf16 fc_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 fc_bf16x2 __attribute__((ext_vector_type(2)));
typedef float fc_floatx2 __attribute__((ext_vector_type(2)));
typedef uint32_t fc_uintx4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 16777216.f, kSplitUnscale = 1.f / (kSplitScale * kSplitScale);      // 2^24, 2^-48

// Two floats to their three parts, packed in pairs.
__device__ __forceinline__ void fc_split2(float a, float b, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    const fc_floatx2 v = {a * kSplitScale, b * kSplitScale};
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, fc_bf16x2));
    fc_floatx2 r = {v[0] - __builtin_bit_cast(float, hi << 16), v[1] - __builtin_bit_cast(float, hi & 0xffff0000u)};
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

// sum += hi * hi, small += the other products, over one stage.  `as`, `bs`: this lane's word of the first part and 32-wide block.
template <int MI, int NI, int A_PLANE, int B_PLANE, class Acc>
__device__ __forceinline__ void fc_split_products(const fc_uintx4 *as, const fc_uintx4 *bs, Acc (&sum)[MI][NI],
                                                  Acc (&small)[MI][NI]) {
    fc_bf16x8 a[3][MI], b[3][NI];
#pragma unroll
    for (int q = 2; q >= 0; q--) {
#pragma unroll
        for (int mi = 0; mi < MI; mi++) a[q][mi] = __builtin_bit_cast(fc_bf16x8, as[q * A_PLANE + mi * 32]);
#pragma unroll
        for (int ni = 0; ni < NI; ni++) b[2 - q][ni] = __builtin_bit_cast(fc_bf16x8, bs[(2 - q) * B_PLANE + ni * 32]);
    }
    constexpr int pa[5] = {2, 1, 0, 1, 0}, pb[5] = {0, 1, 2, 0, 1};
#pragma unroll
    for (int q = 0; q < 5; q++)
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < NI; ni++)
                small[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[q]][mi], b[pb[q]][ni], small[mi][ni], 0, 0, 0);
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
            sum[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][mi], b[0][ni], sum[mi][ni], 0, 0, 0);
}

template <int MI, int NI, class Acc>
__device__ __forceinline__ void fc_zero(Acc (&acc)[MI][NI]) {
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mi][ni][i] = 0.f;
}
// The two sums together, at their true size.
template <int MI, int NI, class Acc>
__device__ __forceinline__ void fc_join(Acc (&acc)[MI][NI], const Acc (&small)[MI][NI]) {
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < NI; ni++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mi][ni][i] = (acc[mi][ni][i] + small[mi][ni][i]) * kSplitUnscale;
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
