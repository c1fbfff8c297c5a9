// fp32 products on the bf16 matrix cores, without losing fp32's precision.
//
// v = v0 + v1 + v2, each a bf16 rounded to nearest from what the ones before leave (3 x 8 significant bits and two signs: nothing of
// the 24 bits is lost down to 2^-108).  Of the nine products of two such sums the six largest are formed; the three left out are
// below 2^-25 of |a b|, half an ulp of an fp32 product.  The matrix cores multiply bf16 pairs exactly and add in fp32; v0 w0 and the five
// corrections go to accumulators of their own, so the small terms are added up at their own scale.
//   Errors against 64 bits, dot products of K elements (2-norm of the error over the result's; normal operands, one sign, products of
//   normals, exponents spread over 2^40), v_mfma_f32_16x16x4_f32 -> this: K = 64 1.06e-7 -> 4.9e-8, 416 2.6e-7 -> 1.1e-7, 1024 4.1e-7 ->
//   1.9e-7; one sign 1.6e-7 -> 1.2e-7 at 416; spread exponents 1.2e-7 -> 1.2e-7 at 416.  (One accumulator for all six: 3.0e-7 at 416, worse
//   than fp32; the three products of two-part sums: 4e-6.)  No bias.
//   Rate: 2.1 PFLOP/s of bf16 measured, 350 TFLOP/s of such products, against 156 of v_mfma_f32_16x16x4_f32.
// An operand that is infinite (or rounds to infinity, above 3.39e38) makes NaN of v1, so every sum it enters comes out NaN; and leading
// parts that were rounded up can overflow where the product of the values does not.  So a tile that holds a sum that is not finite is
// formed again with fp32 instructions (mfma_fp32 below), which gives overflow, infinities and NaNs the meaning they have there.
#pragma once

#include "common.hpp"

namespace kge {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kSplitParts = 3;

// the parts of four consecutive values of a row
__device__ __forceinline__ void split_quad(float4 v, bf16x4 (&p)[kSplitParts])
{
    // (in pairs: v_cvt_pk_bf16_f32 rounds two at a time)
    const f32x2 x[2] = {{v.x, v.y}, {v.z, v.w}};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const bf16x2 a = __builtin_convertvector(x[e], bf16x2);
        const f32x2 r = x[e] - __builtin_convertvector(a, f32x2);
        const bf16x2 b = __builtin_convertvector(r, bf16x2);
        const bf16x2 c = __builtin_convertvector(r - __builtin_convertvector(b, f32x2), bf16x2);
        p[0][2 * e] = a[0], p[0][2 * e + 1] = a[1];
        p[1][2 * e] = b[0], p[1][2 * e + 1] = b[1];
        p[2][2 * e] = c[0], p[2][2 * e + 1] = c[1];
    }
}

// Staged rows: 32 columns of a row as three parts of 64 bytes and 16 bytes of padding, so that 128-bit reads of eight rows at one
// place fall on distinct banks (measured at 128 reads per 563 clocks and CU; 192 bytes a row: 2036).
constexpr int kSplitK = 32;
constexpr int kSplitPitch = kSplitParts * kSplitK + 8;  // bf16s

// one K = 16 step of a 32 x 32 block: lane l holds row l % 32 of its operand, k = 8 (l / 32) .. + 7; receives
// D[row 8 (v / 4) + 4 (l / 32) + v % 4][column l % 32] in v = 0 .. 15
__device__ __forceinline__ floatx16 mfma_bf16(bf16x8 a, bf16x8 b, floatx16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }

// the products of the two operands' parts, smallest first: (part of a, part of b) of step t; the last one is the leading product
constexpr int kSplitTerms = 6;
__device__ constexpr int kTermA[kSplitTerms] = {0, 2, 1, 0, 1, 0}, kTermB[kSplitTerms] = {2, 0, 1, 1, 0, 0};

// ---- the same blocks by fp32 instructions ----
// Whether a sum says nothing about its fp32 value.
__device__ __forceinline__ bool not_finite(float s) { return !(fabsf(s) <= 3.402823466e38f); }

// A K = 2 step of a 32 x 32 block: lane l holds row l % 32 of its operand, k = l / 32; receives what mfma_bf16 gives it.
__device__ __forceinline__ floatx16 mfma_fp32(float a, float b, floatx16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

// Staged rows: 32 columns of a row and 16 bytes of padding (shorter than the three parts').  Eight columns of an A x B block: lane group
// l / 32 takes four of them from 128-bit reads of its rows.
constexpr int kPlainPitch = kSplitK + 4;
static_assert(sizeof(float) * kPlainPitch <= sizeof(__bf16) * kSplitPitch, "fits where the parts stood");
template <int A, int B>
__device__ __forceinline__ void plain_step(const float4 (&av)[A], const float4 (&bv)[B], floatx16 (&acc)[A][B])
{
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
        for (int j = 0; j < B; ++j) {
            acc[i][j] = mfma_fp32(av[i].x, bv[j].x, acc[i][j]);
            acc[i][j] = mfma_fp32(av[i].y, bv[j].y, acc[i][j]);
            acc[i][j] = mfma_fp32(av[i].z, bv[j].z, acc[i][j]);
            acc[i][j] = mfma_fp32(av[i].w, bv[j].w, acc[i][j]);
        }
}

}  // namespace kge
