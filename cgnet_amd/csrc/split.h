// Products of fp32 operands on the half-precision matrix instructions.
//
// v_mfma_f32_16x16x4_f32 holds a SIMD's vector ALUs for its 32 cycles: it and vector instructions take turns.
// v_mfma_f32_16x16x32_f16 takes 16 cycles for eight times the terms and runs beside vector instructions of other waves.  (Probe, eight
// waves a compute unit, half of them vector and half matrix, us: vector half alone 177, fp32 matrix half alone 216, both 383; the same
// with 16-bit matrix instructions 177, 234, 248.)
//
// The left operand's rows and the right operand's columns are scaled by powers of two to a largest entry in [2^14, 2^15), and an entry is
// the sum of two halves h + l (11 + 11 bits and l's sign, the rest rounded off: at most 2^-23 of the entry's leading place or 2^-39 of the
// row's largest entry).  The four products ll + lh + hl + hh are exact and summed in fp32, and the result is scaled back.  Sums of 32
// products of normal numbers against 64 bits, rms error over rms: eight chained fp32 instructions 1.03e-7, this 0.77e-7 (0.88e-7 without
// ll); factors spread log-normally by e^2: 1.11e-7 and 0.66e-7.  The error hardly depends on the number of products, that of the fp32
// chain grows with its root: up to eight (complex) channels the fp32 instructions stay, which are also few then.  Three bfloat16 pieces
// in six products (0.38e-7, no scaling) take half as many bytes again for no less time: lmax 20, 16 channels, B = 32, three layers:
// fp32 6540 us, bfloat16 5660 .. 5830, halves 5840; lmax 11, 12 channels, B = 100: 392, 380, 384.
#pragma once
#include "common.h"

namespace cgnet {

// The 32 places of a product are (output channel, re / im).  Whether halves take the place of fp32 for output channels `t` of the degrees
// 0 .. L: every degree that has any has at least nine.  (gFF against 64 bits, rms, fp32 and halves: 9 channels 8.2e-8 and 8.0e-8, 12
// 9.3e-8 and 7.9e-8, 16 10.6e-8 and 8.1e-8, but 12, 7, 6, 5, 4 ... 3 channels 6.0e-8 and 7.5e-8.)
constexpr int kSplitFrom = 9, kSplitMax = 16;
template <typename Count>
bool split_taken(int L, Count&& t) {
    bool any = false;
    for (int l = 0; l <= L; ++l) {
        if (t(l) != 0 && (t(l) < kSplitFrom || t(l) > kSplitMax)) return false;
        any |= t(l) != 0;
    }
    return any;
}

#ifdef __HIPCC__
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma_half(halfx8 a, halfx8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 split_product(const halfx8 (&a)[2], const halfx8 (&b)[2], f32x4 c = {0.f, 0.f, 0.f, 0.f}) {
    c = mfma_half(a[1], b[1], c);
    c = mfma_half(a[1], b[0], c);
    c = mfma_half(a[0], b[1], c);
    return mfma_half(a[0], b[0], c);
}

// largest modulus of the lane's numbers and of those in the lanes of the other three groups of sixteen
__device__ __forceinline__ float split_largest(const float (&x)[8]) {
    float m = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) m = fmaxf(m, fabsf(x[q]));
    m = fmaxf(m, __shfl_xor(m, 16));
    return fmaxf(m, __shfl_xor(m, 32));
}
// The exponent an operand's row is scaled by (the result's scale: 2^-e).  Below 2^-110 a row keeps its absolute error.
__device__ __forceinline__ int split_exponent(float largest) {
    return 15 - max(-110, __builtin_amdgcn_frexp_expf(largest));
}
__device__ __forceinline__ float split_scale(int e) { return __builtin_amdgcn_ldexpf(1.f, -e); }
__device__ __forceinline__ void split8(const float (&x)[8], int e, halfx8 (&p)[2]) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const float s = __builtin_amdgcn_ldexpf(x[q], e);
        p[0][q] = (_Float16)s;
        p[1][q] = (_Float16)(s - (float)p[0][q]);
    }
}
#endif

}  // namespace cgnet
