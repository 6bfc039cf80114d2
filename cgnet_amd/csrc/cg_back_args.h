// What the host and the kernel of the backward by pairs share: arguments, LDS layout, variants.
#pragma once
#include "cg_back.h"

namespace cgnet {

struct BackArgs {
    const float2* F;
    const float2* gFF;             // memory source
    const float* Go;               // layer source: packed gO, packed weights
    const float* W;
    const BackGenPair* gp;
    const float* coef;
    const BackPair* pairs;
    const BackUnit* units;
    float2* part;
    int nF, nFF, go_chunk, go_degree, nGo, P, grid0, B, nunits, lds_wave;
};

// LDS of a wave (floats): sums [rows][kBackPitch] complex | a row of zeros | two buffers of nrows rows of degree l1 between zeros.
// Row r stands for m1 = first M + l2 - 16 nt + 1 + r.
constexpr int kBackPitch = 20;                 // complex entries per m1 of the LDS sums: sixteen columns, rows four apart fall on other banks
__host__ __device__ inline int back_rows(int nch, int nt) { return 8 * nch + 16 * nt - 1; }
__host__ __device__ inline int back_row_pitch(int rows) { return rows | 1; }
__host__ __device__ inline int back_lds_floats(int nch, int nt, int nrows) {
    const int rows = back_rows(nch, nt);
    return (2 * (rows * kBackPitch + (2 * nrows + 1) * back_row_pitch(rows)) + 3) & ~3;
}

// a variant's kernel for the layer source with so many pairs of steps (0: memory source), and its launch
#define CGNET_BACK_DECLARE(V)              \
    const void* back_kernel_##V(int pairs); \
    void back_launch_##V(int pairs, dim3 grid, size_t lds, hipStream_t s, const BackArgs& a);
CGNET_BACK_DECLARE(0)
CGNET_BACK_DECLARE(1)
CGNET_BACK_DECLARE(2)
CGNET_BACK_DECLARE(3)
constexpr int kBackThreads = 64 * kBackWaves;

}  // namespace cgnet
