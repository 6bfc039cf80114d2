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
    int nF, nFF, go_chunk, go_degree, go_scales, lanes, nGo, P, grid0, B, nunits, lds_wave;
};

// LDS of a wave (floats): sums [rows][kBackPitch] complex | a row of zeros | nbuf buffers of nrows rows of degree l1 between zeros (two
// where a unit has several tiles: the next one's rows are fetched ahead).  Row r stands for m1 = first M + l2 - 16 nt + 1 + r.  The row
// of zeros begins in the unused columns of the last sum and ends in the first entry of a fragment row, which stands for no m1
// (16 nt - 1 - l2 - l1 + lm >= 16 nt - 1 - 2 l2 > 0 entries lie before m1 = -l1): with three rows t1 at lmax 20..23 this is what lets two
// work-groups share a compute unit (81 920 bytes each).
constexpr int kBackPitch = 20;                 // complex entries per m1 of the LDS sums: sixteen columns, rows four apart fall on other banks
constexpr int kBackSpare = kBackPitch - 16;    // columns of a sum that nothing is added to
__host__ __device__ inline int back_rows(int nch, int nt) { return 8 * nch + 16 * nt - 1; }
__host__ __device__ inline int back_row_pitch(int rows) { return rows; }     // (odd)
__host__ __device__ inline int back_lds_floats(int nch, int nt, int nrows, int nbuf) {
    const int rows = back_rows(nch, nt);
    return (2 * (rows * kBackPitch - kBackSpare + (nbuf * nrows + 1) * back_row_pitch(rows) - 1) + 3) & ~3;
}

// a variant's kernel for a source of the product's gradient (cg_back.h), and its launch
#define CGNET_BACK_DECLARE(V)              \
    const void* back_kernel_##V(int source); \
    void back_launch_##V(int source, dim3 grid, size_t lds, hipStream_t s, const BackArgs& a);
CGNET_BACK_DECLARE(0)
CGNET_BACK_DECLARE(1)
CGNET_BACK_DECLARE(2)
CGNET_BACK_DECLARE(3)
constexpr int kBackThreads = 64 * kBackWaves;

}  // namespace cgnet
