// Products of fp32 operands on the 16-bit matrix instructions.
//
// v_mfma_f32_16x16x4_f32 holds a SIMD's vector ALUs for its 32 cycles: it and vector instructions take turns.
// v_mfma_f32_16x16x32_bf16 takes 16 cycles for eight times the terms, of which vector instructions of other waves hide four
// (profiles/matrix_vector_issue.txt).
//
// An operand is the sum of three bfloat16 pieces h + m + l, which hold its 24 bits, and six of the nine products (ml, lm and ll, together
// at most 2^-23 of the product and mostly far less, are left out) are summed in fp32.  bfloat16 has the exponents of fp32: an entry keeps its
// bits whatever lies beside it, down to 2^-110 (below, an absolute error of 2^-134).  gO, whose size follows the loss, is scaled by a power
// of two where its largest entry is below 2^-16, to [2^-17, 2^-16): entries down to 2^-93 of that one keep their bits, and products with
// weights of any size stay in range until the result is scaled back.
// gFF against 64 bits (rms, lmax 11, whether or not the output channels are spread over six decades): 9 channels 7.8e-8 by fp32 instructions,
// 3.5e-8 by pieces, 12 channels 8.9e-8 and 3.6e-8, 16 channels 10.2e-8 and 3.8e-8.
// Backward by pairs (cg_back_kernel.h), fp32 instructions -> pieces, us: lmax 20, 16 channels, B = 32: 2136 -> 1976; gFF alone, lmax 11, 16
// channels, B = 64: 252 -> 183.  Two f16 pieces with a scale for each row and column took 1921, but lost what lay 2^16 and more below the
// largest of its row or column: output channels spread over ten decades, with weights and gO that balance each other, came back with an
// error of 3e-3.
#pragma once
#include "common.h"

namespace cgnet {

// The 32 places of a product are (output channel, re / im).  Whether pieces take the place of fp32 for output channels `t` of the degrees
// 0 .. L: every degree that has any has at least thirteen.  They replace seven or eight fp32 instructions there, five or six at nine to
// twelve channels, and operands half as large again there, twice as large at twelve.  Kernels of a training step over lmax 2..23, 1..64 samples, fp32 -> pieces:
//   13 .. 16 channels  layer 0.98 of the time (215 shapes, two more than 3 % slower: 96 -> 99 us), gFF alone 0.90 (8 of 215 more than 5 % slower, up
//                      to four samples: 22 -> 25 us, 125 -> 135)
//   10 .. 12 channels  layer 1.01 (35 of 262 more than 3 % slower, 507 -> 542 us at lmax 20, 16 -> 12 channels, one sample), gFF alone 0.99 (75 of
//                      262 more than 5 % slower, 28.6 -> 35.2 us at lmax 18, 10 channels, one sample)
//   up to eight        layer of 5 channels at lmax 11, B = 100: 278 -> 292 us, of 8 624 -> 650
// Above degree 23, where there is no backward by pairs either, the stand-alone kernel would split gO again for every tile of channels.
constexpr int kPieces = 3;
constexpr int kSplitFrom = 13, kSplitMax = 16, kSplitMaxL = 23;
template <typename Count>
bool split_taken(int L, Count&& t) {
    if (L > kSplitMaxL) return false;
    bool any = false;
    for (int l = 0; l <= L; ++l) {
        if (t(l) != 0 && (t(l) < kSplitFrom || t(l) > kSplitMax)) return false;
        any |= t(l) != 0;
    }
    return any;
}

#ifdef __HIPCC__
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma_piece(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// a: gO, b: weights, small products first
__device__ __forceinline__ f32x4 split_product(const bf16x8 (&a)[kPieces], const bf16x8 (&b)[kPieces]) {
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
    c = mfma_piece(a[2], b[0], c);
    c = mfma_piece(a[0], b[2], c);
    c = mfma_piece(a[1], b[1], c);
    c = mfma_piece(a[1], b[0], c);
    c = mfma_piece(a[0], b[1], c);
    return mfma_piece(a[0], b[0], c);
}

// largest modulus of the lane's numbers and of those in the lanes of the other three groups of sixteen
__device__ __forceinline__ float split_largest(const float (&x)[8]) {
    float m = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) m = fmaxf(m, fabsf(x[q]));
    m = fmaxf(m, __shfl_xor(m, 16));
    return fmaxf(m, __shfl_xor(m, 32));
}
// The exponent gO is scaled by; its power of two and the one that scales back are normal numbers.  (A lone zero: any.)
__device__ __forceinline__ int split_exponent(float largest) {
    const int f = __builtin_amdgcn_frexp_expf(largest);            // largest < 2^f
    return min(max(-16 - f, min(0, 127 - f)), 126);                // (at f = 128 a first piece could round to infinity)
}
__device__ __forceinline__ float split_scale(int e) { return __builtin_amdgcn_ldexpf(1.f, e); }

__device__ __forceinline__ void split8(const float (&x)[8], float scale, bf16x8 (&p)[kPieces]) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    u32x4 u[kPieces];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        f32x2 r = {x[2 * q] * scale, x[2 * q + 1] * scale};
#pragma unroll
        for (int k = 0; k < kPieces; ++k) {
            const unsigned h = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
            u[k][q] = h;
            r.x -= __uint_as_float(h << 16);                       // exact
            r.y -= __uint_as_float(h & 0xffff0000u);
        }
    }
#pragma unroll
    for (int k = 0; k < kPieces; ++k) p[k] = __builtin_bit_cast(bf16x8, u[k]);
}
// Weights, unscaled.  One that would round to infinity has its first piece cut off instead.  One that is not finite lies in the third
// piece, which meets the first of gO alone, with its sign: pieces of either sign beside it would make inf - inf of what is an infinity in a
// chain of fp32 products.
__device__ __forceinline__ void split8_weights(const float (&x)[8], bf16x8 (&p)[kPieces]) {
    float y[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) y[q] = fabsf(x[q]) >= 0x1p127f ? 0.f : x[q];
    split8(y, 1.f, p);
#pragma unroll
    for (int q = 0; q < 8; ++q)
        if (!(fabsf(x[q]) < 0x1p127f)) {
            const float h = __uint_as_float(__float_as_uint(x[q]) & 0xffff0000u), r = x[q] - h;
            const float m = __uint_as_float(__float_as_uint(r) & 0xffff0000u);
            const bool finite = fabsf(x[q]) <= 0x1.fffffep127f;
            p[0][q] = (__bf16)(finite ? h : 0.f);
            p[1][q] = (__bf16)(finite ? m : 0.f);
            p[2][q] = (__bf16)(finite ? r - m : x[q]);
        }
}
#endif

}  // namespace cgnet
