// Backward of the Clebsch-Gordan product organised by pairs of input degrees (cg_back.hip): types shared with the plans.
#pragma once
#include <vector>

#include "split.h"

namespace cgnet {

struct PairTriple;

constexpr int kBackMaxL = 23;      // 2L+1 <= 48 rows: three row tiles of sixteen values of m2
constexpr int kBackMaxTau = 16;    // channels of degree l2: the columns of a tile
constexpr int kBackNL = 16;        // output degrees of a pair, in groups of four
constexpr int kBackChunks = 6;     // chunks of eight values of M = m1 + m2
constexpr int kBackWaves = 4;      // waves of a work-group: samples of the same unit
constexpr int kBackMaxRows = 8;    // rows t1 of a tile at most (their fragments are staged twice)

// A pair (l1, l2) with its output degrees, largest first (at most kBackNL: more make a pair of their own).  Its tau1 x tau2 channels
// (t1, t2) are cut into tiles of ncol columns; the tiles of a unit lie tstep apart, so that a column has the same t2 in all of them.
struct BackPair {
    int l1, l2, tau1, tau2;
    int nl, nks;                   // output degrees, groups of four
    int nt;                        // row tiles of sixteen m2
    int ncol, ntiles, tstep;
    int nrows;                     // rows t1 that a tile touches, at most
    int c0, nch;                   // chunks of eight M: the first, how many
    int offF1, offF2;              // complex offsets of the two degrees inside a sample's F
    int coef;                      // float offset of the packed coefficients: [M - first][group][row tile][64]
    int steps[kBackChunks];        // per chunk, four bits per M: groups with a degree >= |M|
    int tiles[kBackChunks];        // per chunk, four bits per M: row tiles that hold a valid m2
    int degs[kBackChunks];         // per chunk: output degrees that reach into it
    int l[kBackNL], cg[kBackNL];   // output degrees, float offsets of their tables
    int offFF[kBackNL];            // complex offset inside a sample's gFF of channel (0, 0)
    int inv_tau2, inv_M1, inv_M2;  // ceil(2^16 / tau2), ceil(2^20 / (2 l1 + 1)), ceil(2^20 / (2 l2 + 1))
    int ends;                      // bit 0 / 1: the first / last channel of a degree is the first / last of a sample's product
    int nbuf;                      // buffers of F1 rows
    unsigned l8[kBackNL / 4];      // the output degrees again, a byte each
};

// One wave's share of a pair: tiles tile0, tile0 + tstep, ...  Its partial gradients inside a sample's: nrows rows of degree l1 per
// tile at p1off, all channels of degree l2 at p2off (complex offsets).
struct BackUnit { int pair, tile0, ntiles, p1off, p2off; };

// A cut of all pairs into units for a range of batch sizes.
struct BackLevel {
    int least_B = 1;               // taken from this batch on (levels from coarse to fine, the last from one sample on)
    std::vector<BackUnit> units;   // longest first
    BackUnit* d_units = nullptr;
    int* d_combine = nullptr;      // meta of cg_backward_rows_kernel
    int P = 0;                     // complex entries of one sample's partial gradients
};

struct BackSet {
    std::vector<BackPair> pairs;
    std::vector<BackLevel> levels;
    unsigned char* d_tables = nullptr;     // pairs, coefficient map, units and combine metas: one allocation
    BackPair* d_pairs = nullptr;
    int2* d_coefmap = nullptr;             // per block of the coefficient packing: pair, M - first
    int ncoefmap = 0;
    size_t coef_floats = 0;
    int grid0 = 0;                         // M of the first value of chunk 0 (chunks of all pairs lie on one grid)
    int nchunks = 0;                       // chunks of the grid
    int variant = 0;                       // kernel variant (groups x row tiles)
    size_t lds = 0;                        // LDS bytes of a work-group
    // of one sample: 16 x 16 blocks of H that the vector ALUs multiply, tiles of channels, multiply-adds of one gradient triple by
    // triple
    double blocks = 0., tiles = 0., macs = 0.;
    bool ok() const { return !pairs.empty(); }
};

// Inside the layer the gradient of the product is made from packed weights and packed gO, both in lane order.
struct BackGenPair {
    int w, wtile;                  // float offset of the pair's first tile, floats of a tile
};
struct BackGenW {                  // of a (pair, degree): what packing its weights needs to know
    int chan0, nch;                // the triple's channels inside degree l: first, count
    int tO, cumW, K, cumT;         // degree l: output channels, complex offset of its weights, mid channels, first of them among all
    int source, at;                // BackLink::source, float offset of the first tile's operands
    int ncol, ntiles, wtile;       // columns of a tile, tiles, floats from one tile to the next
};

// Where the kernel's gradient of the product comes from: memory; packed gO and weights, multiplied in one to four pairs of steps (of
// four output channels) of v_mfma_f32_16x16x4_f32, or as pieces (split.h: floats of an operand, of the scales of a chunk of eight M).
constexpr int kBackMemory = 0, kBackSplit = 5;
constexpr int kBackOperand = 256 * kPieces, kBackScales = 8;

struct BackLink {
    bool ok = false;
    unsigned char* d_tables = nullptr;
    BackGenPair* d_gp = nullptr;
    int2* d_degs = nullptr;        // per degree: cumO, t_O
    int* d_reach = nullptr;        // per (degree, output degree): the largest degree of the other fragment, -1: no such pair
    BackGenW* d_gens = nullptr;
    int ngens = 0, ndeg = 0;
    int source = 0;                // by the degree with most outputs, pieces where the one with fewest allows it
    size_t w_floats = 0;           // packed weights
    int go_degree = 0, go_flags = 0, go_floats = 0;    // packed gO of a degree, of a sample up to its flags, with scales and flags
    int lanes = 64;                // lanes that hold places of output channels
    int nO = 0;                    // complex entries of one sample's layer output
    int most_B = 0;                // the largest batch it is taken for where there is another route
};

#ifdef __HIPCC__
// The coefficients of a pair for one M, by one work-group: [group of four degrees][row tile][lane (degree, m2)]; zeros where M is
// no value of the degree or M - m2 none of degree l1, whatever the caller's table holds there.
__device__ __forceinline__ void pack_coef_back_block(const float* __restrict__ CG, const BackPair* __restrict__ pairs, int2 which,
                                                     int grid0, float* __restrict__ coef) {
    const BackPair& p = pairs[which.x];
    const int x = which.y, M = grid0 + 8 * p.c0 + x, M2 = 2 * p.l2 + 1;
    const int nk = (p.steps[x >> 3] >> (4 * (x & 7))) & 15;
    float* dst = coef + p.coef + x * p.nks * p.nt * 64;
    for (int e = threadIdx.x; e < nk * p.nt * 64; e += blockDim.x) {
        const int lane = e & 63, blk = e >> 6, g = blk / p.nt, rt = blk - g * p.nt;
        const int q = 4 * g + (lane >> 4), m = 16 * rt + (lane & 15), m1 = M - (m - p.l2);
        float v = 0.f;
        if (q < p.nl && m < M2 && m1 >= -p.l1 && m1 <= p.l1) {
            const int l = p.l[q];
            if (M >= -l && M <= l) v = CG[p.cg[q] + (M + l) * M2 + m];
        }
        dst[e] = v;
    }
}

// The weights of a (pair, degree) as right operands, tiles wave, wave + 4, ...: W / max(eps, std) of the column's channel, zero past t_O
// and past the tile's channels.  As pieces: per tile [degree][piece][lane (k, column)] of eight k = (output channel, re / im).  For fp32
// steps: per tile and group of four degrees
// [pair of steps][pair of degrees][lane (k, column)][degree][step].
__device__ __forceinline__ void pack_w_back_wave(const float2* __restrict__ W, const float* __restrict__ stds, float eps,
                                                 const BackGenW& g, int wave, int lane, float* __restrict__ Wp) {
    const int j = lane & 15, kk = lane >> 4;
    for (int tile = wave; tile < g.ntiles; tile += 4) {
        const int cl = tile * g.ncol + j;
        const bool on = j < g.ncol && cl < g.nch;
        const int c = g.chan0 + cl;
        const float r = (on && stds) ? fmaxf(eps, stds[g.cumT + c]) : 1.f;
        float* dst = Wp + g.at + (size_t)tile * g.wtile + 4 * lane;
        if (g.source == kBackSplit) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int to = 4 * kk + e;
                float2 w = make_float2(0.f, 0.f);
                if (on && to < g.tO) {
                    w = W[g.cumW + (size_t)to * g.K + c];
                    if (stds) w = make_float2(w.x / r, w.y / r);
                }
                v[2 * e] = w.x;
                v[2 * e + 1] = w.y;
            }
            bf16x8 p[kPieces];
            split8_weights(v, p);
#pragma unroll
            for (int k = 0; k < kPieces; ++k) *reinterpret_cast<bf16x8*>(dst + 256 * k) = p[k];
            continue;
        }
        for (int s = 0; s < g.source; ++s) {
            float v[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int k = 4 * (2 * s + e) + kk, to = k >> 1;
                v[e] = 0.f;
                if (on && to < g.tO) {
                    const float2 w = W[g.cumW + (size_t)to * g.K + c];
                    v[e] = (k & 1) ? w.y : w.x;
                    if (stds) v[e] = v[e] / r;
                }
            }
            *reinterpret_cast<float2*>(dst + 512 * s) = make_float2(v[0], v[1]);
        }
    }
}
#endif

}  // namespace cgnet
