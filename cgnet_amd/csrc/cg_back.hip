// Backward of the Clebsch-Gordan product organised by pairs of input degrees: plans, packing kernels and launches.  The kernel
// and what it does: cg_back_kernel.h.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <memory>
#include <numeric>

#include "cg_back_args.h"
#include "internal.h"

namespace cgnet {
namespace {

// The coefficients of all pairs, one work-group per (pair, M).
__global__ void __launch_bounds__(256)
pack_coef_back_kernel(const float* __restrict__ CG, const BackPair* __restrict__ pairs, const int2* __restrict__ map, int grid0,
                      float* __restrict__ coef) {
    pack_coef_back_block(CG, pairs, map[blockIdx.x], grid0, coef);
}

__device__ __forceinline__ bool finite(float2 z) {
    return (__float_as_uint(z.x) & 0x7f800000u) != 0x7f800000u && (__float_as_uint(z.y) & 0x7f800000u) != 0x7f800000u;
}

// Packed gO of the layer source, k = (channel, re / im); zero past the degree's channels and values, and in the place of entries that are
// not finite; behind it a flag per (chunk of eight M, degree): whether it has such entries.  degs: per degree cumO, t_O.
struct GoEntries {
    const float2* src;
    int l, tO, x;
    bool odd = false;
    __device__ __forceinline__ GoEntries(const float2* gO, int2 d, int l, int M) : src(gO + d.x), l(l), tO(d.y), x(M + l) {}
    __device__ __forceinline__ float2 operator()(int to) {
        if (to >= tO || x < 0 || x > 2 * l) return make_float2(0.f, 0.f);
        const float2 z = src[to * (2 * l + 1) + x];
        if (finite(z)) return z;
        odd = true;
        return make_float2(0.f, 0.f);
    }
};

// For fp32 steps: [chunk][degree][step][lane (k, (M, re / im))].  A work-group takes a (chunk, degree) of a sample.
__global__ void __launch_bounds__(64)
pack_go_back_kernel(const float2* __restrict__ gO, const int2* __restrict__ degs, float* __restrict__ Go, int ndeg, int pairs, int grid0,
                    int nO, int nGo) {
    const int l = (int)blockIdx.x % ndeg, c = (int)blockIdx.x / ndeg;
    const int lane = threadIdx.x, i = lane & 15, kk = lane >> 4, r = i & 1;
    GoEntries entry(gO + (size_t)blockIdx.y * nO, degs[l], l, grid0 + 8 * c + (i >> 1));
    float* const sample = Go + (size_t)blockIdx.y * nGo;
    float* dst = sample + (size_t)blockIdx.x * 128 * pairs + lane;
    for (int s = 0; s < 2 * pairs; ++s) {
        const int k = 4 * s + kk, sel = k & 1;
        const float2 z = entry(k >> 1);
        dst[64 * s] = (r == sel) ? (r ? -z.x : z.x) : z.y;
    }
    const int odd = __any(entry.odd);
    if (lane == 0) reinterpret_cast<int*>(sample)[(size_t)gridDim.x * 128 * pairs + blockIdx.x] = odd;
}

// As pieces: [degree][chunk][piece][lane (k, (M, re / im))] of eight k, then [chunk][M] scales: the degrees share one, so that the pair
// kernel holds it for a chunk (a scale for each degree: 74 instead of 46 registers spilled at lmax 8..11, layer of 12 channels at lmax 11,
// B = 100: 1199 us a step instead of 1029).  A work-group takes a chunk of a sample, its waves the degrees in turn.
constexpr int kPackGoWaves = 8;
__global__ void __launch_bounds__(64 * kPackGoWaves)
pack_go_back_split_kernel(const float2* __restrict__ gO, const int2* __restrict__ degs, float* __restrict__ Go, int ndeg, int grid0, int nO,
                          int nGo) {
    __shared__ float s_top[kPackGoWaves][16];
    const int c = (int)blockIdx.x, nchunks = (int)gridDim.x, places = nchunks * ndeg;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = lane & 15, kk = lane >> 4, r = i & 1;
    float* const sample = Go + (size_t)blockIdx.y * nGo;
    int* const flags = reinterpret_cast<int*>(sample) + kBackOperand * places + kBackScales * nchunks + c * ndeg;
    constexpr int kMost = (kBackMaxL + kPackGoWaves) / kPackGoWaves;       // degrees of a wave
    float v[kMost][8], top = 0.f;
#pragma unroll
    for (int n = 0; n < kMost; ++n) {
        const int l = wave + n * kPackGoWaves;
        if (l >= ndeg) break;
        GoEntries entry(gO + (size_t)blockIdx.y * nO, degs[l], l, grid0 + 8 * c + (i >> 1));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float2 z = entry(4 * kk + e);
            v[n][2 * e] = r ? z.y : z.x;
            v[n][2 * e + 1] = r ? -z.x : z.y;
        }
        top = fmaxf(top, split_largest(v[n]));
        const int odd = __any(entry.odd);
        if (lane == 0) flags[l] = odd;
    }
    if (lane < 16) s_top[wave][lane] = top;                        // (the same for both columns of an M)
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kPackGoWaves; ++w) top = fmaxf(top, s_top[w][i]);
    const int e = split_exponent(top);
    if (wave == 0 && lane < 16 && r == 0) sample[kBackOperand * places + kBackScales * c + (i >> 1)] = split_scale(-e);
    const float scale = split_scale(e);
#pragma unroll
    for (int n = 0; n < kMost; ++n) {
        const int l = wave + n * kPackGoWaves;
        if (l >= ndeg) break;
        bf16x8 p[kPieces];
        split8(v[n], scale, p);
        bf16x8* dst = reinterpret_cast<bf16x8*>(sample + (size_t)kBackOperand * (l * nchunks + c)) + lane;
#pragma unroll
        for (int k = 0; k < kPieces; ++k) dst[64 * k] = p[k];
    }
}

// What cg_backward_rows_kernel looks at where something is not finite.
struct BackTerms {
    const BackPair* pairs;         // memory source
    const float2 *F, *gFF;
    const float* coef;
    const float2* gO;              // layer source
    const int* odd;                // ... the flags of pack_go_back_kernel
    const int2* degs;
    const int* reach;              // ... per (degree l, degree d of gO): the largest degree of a fragment between them, -1: none
    int nFF, nO, nGo, nodd, ndeg, grid0;
};

// Entry m of row t of a degree: its share from some of a pair's tiles, term by term.  which: pair and whether the degree is the pair's
// l2; tiles: the first, how many << 16.
__device__ float2 back_share(const BackTerms& a, int b, int nF, int t, int m, int which, int tiles) {
    const BackPair& p = a.pairs[which >> 1];
    const bool second = which & 1;
    const int n = second ? p.tau1 : p.tau2, lo = second ? p.l1 : p.l2;
    const float2* other = a.F + (size_t)b * nF + (second ? p.offF1 : p.offF2);
    const float2* G = a.gFF + (size_t)b * a.nFF;
    float2 s = make_float2(0.f, 0.f);
    for (int o = 0; o < n; ++o) {
        const int c = second ? o * p.tau2 + t : t * p.tau2 + o, k = c / p.ncol - (tiles & 0xffff);
        if (k < 0 || k >= (tiles >> 16) * p.tstep || k % p.tstep) continue;
        for (int mo = max(-lo, -p.l[0] - m); mo <= min(lo, p.l[0] - m); ++mo) {
            const int M = m + mo, m2 = p.l2 + (second ? m : mo);
            const float* coef = a.coef + p.coef + ((M - a.grid0 - 8 * p.c0) * p.nks * p.nt + (m2 >> 4)) * 64 + (m2 & 15);
            float2 h = make_float2(0.f, 0.f);
#pragma unroll 4
            for (int q = 0; q < p.nl; ++q) {
                const int l = p.l[q];
                if (abs(M) > l) break;
                const float2 g = G[p.offFF[q] + c * (2 * l + 1) + M + l];
                const float v = coef[(q >> 2) * p.nt * 64 + 16 * (q & 3)];
                h.x += v * g.x;
                h.y += v * g.y;
            }
            const float2 z = other[o * (2 * lo + 1) + lo + mo];
            s.x += h.x * z.x + h.y * z.y;
            s.y += h.y * z.x - h.x * z.y;
            if (!finite(s)) return s;                              // and stays so
        }
    }
    return s;
}

// Whether an entry of the sample's gO that is not finite is in the gradient of entry m of degree l: it is in G of every channel.
__device__ bool back_reached(const BackTerms& a, int b, int l, int m) {
    for (int k = 0; k < a.nodd; ++k) {
        if (!a.odd[(size_t)b * a.nGo + k]) continue;
        const int d = k % a.ndeg, M0 = a.grid0 + 8 * (k / a.ndeg), far = a.reach[l * a.ndeg + d];
        const float2* g = a.gO + (size_t)b * a.nO + a.degs[d].x + d;
        for (int M = max(max(-d, M0), m - far); M <= min(min(d, M0 + 7), m + far); ++M)
            for (int to = 0; to < a.degs[d].y; ++to)
                if (!finite(g[to * (2 * d + 1) + M])) return true;
    }
    return false;
}

// Input gradient from the units' partial ones: a row's shares added in the order of its list.
// The pair kernel multiplies places that stand for no value of m, no degree or no channel by zero coefficients, and zero times
// infinity is no zero.  An entry of the gradient that comes in and is not finite still reaches what depends on it and nothing else: from
// memory, a share that is not finite is added up again term by term; the layer's gO is packed without such entries, and what depends
// on them is made NaN here.  (Masks in the pair kernel itself, even as a second pass off its hot path, cost it 1 .. 6 %: more registers
// to spill, and a check per unit.)  Whole backward at lmax 20, 16 channels, B = 8: inside the layer 0.8 ms whatever gO holds; from memory
// 0.7 ms where all is finite or nothing is, 2.8 with one infinity in each sample, 9.4 where some sums of every row are too large.
// meta: [L+2] cumF | [L+2] first row of a degree | [rows + 1] list begin | offsets of the shares | which, tiles of back_share
__global__ void __launch_bounds__(256)
cg_backward_rows_kernel(const float2* __restrict__ part, float2* __restrict__ gF, const int* __restrict__ meta, int L, int nF, int P,
                        int B, BackTerms terms) {
    __shared__ int s_tab[kMaxLookup];
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int b = (int)(idx / nF), e = (int)(idx % nF);
    const int* cum_rows = meta + (L + 2);
    const int* begin = cum_rows + (L + 2);
    const int* at = begin + cum_rows[L + 1] + 1;
    const int lane = threadIdx.x & 63, b0 = __builtin_amdgcn_readfirstlane(b), b1 = min(__builtin_amdgcn_readlane(b, 63), B - 1);
    // flags of the wave's samples: the first 64 are fetched here and looked at behind the sums
    const int nodd = terms.nodd, flags = (b1 - b0 + 1) * nodd;
    auto flag = [&](int k) { return terms.odd[(size_t)(b0 + k / nodd) * terms.nGo + k % nodd]; };
    int odd = lane < flags ? flag(lane) : 0;
    const int l = lookup_in_group(L + 1, e, [&](int k) { return meta[k]; }, s_tab);
    const int M = 2 * l + 1, rel = e - s_tab[l], t = rel / M, x = rel - t * M;
    const int row = cum_rows[l] + t, k0 = begin[row], k1 = b < B ? begin[row + 1] : k0;     // (lanes past the end fetch flags)
    const float2* from = part + (size_t)b * P + x;
    float2 s = make_float2(0.f, 0.f);
#pragma unroll 8
    for (int k = k0; k < k1; ++k) {
        const float2 v = from[at[k]];
        s.x += v.x;
        s.y += v.y;
    }
    if (terms.gFF && __builtin_expect(!finite(s), 0)) {
        const int* which = at + begin[cum_rows[L + 1]];
        s = make_float2(0.f, 0.f);
        for (int k = k0; k < k1 && finite(s); ++k) {
            float2 v = from[at[k]];
            if (!finite(v)) v = back_share(terms, b, nF, t, x - l, which[2 * k], which[2 * k + 1]);
            s.x += v.x;
            s.y += v.y;
        }
    }
    if (nodd) {
        for (int k = lane + 64; k < flags; k += 64) odd |= flag(k);
        if (__builtin_expect(__any(odd), 0) && b < B && back_reached(terms, b, l, x - l)) s = make_float2(__builtin_nanf(""), __builtin_nanf(""));
    }
    if (b < B) gF[idx] = s;
}

// Packed weights of the layer source, one work-group of four waves per (pair, degree).
__global__ void __launch_bounds__(256)
pack_w_back_kernel(const float2* __restrict__ W, const float* __restrict__ stds, float eps, const BackGenW* __restrict__ gens,
                   float* __restrict__ Wp) {
    pack_w_back_wave(W, stds, eps, gens[blockIdx.x], (int)(threadIdx.x >> 6), threadIdx.x & 63, Wp);
}

constexpr int kVariants = 4;                       // kernel variants, by the largest degree
constexpr int kVariantL[kVariants] = {7, 11, 15, kBackMaxL};
// Groups of four output degrees: the smallest number that holds all of a pair, up to lmax 15.  Above it that took 256 registers, 177
// of them spilled, at six groups; a pair of more than sixteen degrees is cut, its smaller ones make a pair of their own that spans few M
// (layer, lmax 20, 16 channels, B = 32: 2.39 -> 2.18 ms, five groups 2.28, three 2.27; from memory at B = 16: 1.54 -> 1.14 ms).  Where
// all fit, cutting only repeats the vector half (lmax 11, 12 channels, B = 100, cut at two groups: 1.07 times as long; lmax 15, 16 channels,
// B = 64, cut at three: 1.08).
constexpr int kVariantKS[kVariants] = {2, 3, 4, 4};

const void* variant_kernel(int v, int source) {
    return v == 0 ? back_kernel_0(source) : v == 1 ? back_kernel_1(source) : v == 2 ? back_kernel_2(source) : back_kernel_3(source);
}

int launch_back(const BackSet& set, const BackLevel& lv, int source, BackArgs a, BackTerms t, float* d_gF, int L, hipStream_t s) {
    a.pairs = set.d_pairs; a.units = lv.d_units; a.P = lv.P; a.grid0 = set.grid0;
    a.lds_wave = (int)(set.lds / (4 * kBackWaves));
    a.nunits = (int)lv.units.size();
    const int quads = (a.B + kBackWaves - 1) / kBackWaves;
    CGNET_REQUIRE((long long)a.nunits * quads < (1LL << 31), CGNET_ERR_UNSUPPORTED, "%d units x %d sample groups exceed the grid limit",
                  a.nunits, quads);
    const dim3 grid((unsigned)(a.nunits * quads));
    auto* launch = set.variant == 0 ? back_launch_0 : set.variant == 1 ? back_launch_1 : set.variant == 2 ? back_launch_2 : back_launch_3;
    launch(source, grid, set.lds, s, a);
    CGNET_HIP(hipGetLastError());
    t.pairs = set.d_pairs; t.grid0 = set.grid0;
    const size_t n = (size_t)a.nF * a.B;
    CGNET_LAUNCH(cg_backward_rows_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a.part, (float2*)d_gF, lv.d_combine, L,
                 a.nF, lv.P, a.B, t);
    CGNET_HIP(hipGetLastError());
    return CGNET_OK;
}

}  // namespace

const BackLevel& back_level(const BackSet& set, int B) {
    for (const BackLevel& lv : set.levels)
        if (B >= lv.least_B) return lv;
    return set.levels.back();
}

int back_most_batch(const BackSet& set, int L, int nFF, int ntasks, const BackRule& rule) {
    const double more = 1e-4 * (rule.block * set.blocks + rule.tile * set.tiles - rule.mac * set.macs - rule.entry * nFF - rule.task * ntasks);
    const double most = rule.start + rule.start_L2 * L * L;
    return more <= 0. || most / more >= 1e6 ? INT32_MAX : (int)(most / more);
}

void free_back_set(BackSet* set) {
    if (set->d_tables) (void)hipFree(set->d_tables);
    *set = BackSet();
}

int build_back_set(const std::vector<PairTriple>& triples, const std::vector<int>& t_F, const std::vector<int>& cumF, int L, int nFF,
                   BackSet* out) {
    free_back_set(out);
    if (L > kBackMaxL || nFF < 2 || nFF >= 1 << 28) return CGNET_OK;       // (32-bit byte offsets in a sample, sixteen bytes a load)
    for (int t : t_F)
        if (t > kBackMaxTau) return CGNET_OK;
    // triples by pair, largest output degree first; the n-th repetition of a triple goes into a list of its own
    std::vector<std::array<int, 5>> order;                                     // l1, l2, repetition, -l, triple
    for (size_t k = 0; k < triples.size(); ++k)
        if (t_F[triples[k].l1] > 0 && t_F[triples[k].l2] > 0) order.push_back({triples[k].l1, triples[k].l2, 0, -triples[k].l, (int)k});
    if (order.empty()) return CGNET_OK;
    std::sort(order.begin(), order.end());
    for (size_t k = 1; k < order.size(); ++k)
        if (order[k][0] == order[k - 1][0] && order[k][1] == order[k - 1][1] && order[k][3] == order[k - 1][3])
            order[k][2] = order[k - 1][2] + 1;
    std::sort(order.begin(), order.end());
    // The grid of chunks: of the eight places of its origin the one with the fewest chunks in all.
    int best = -1;
    for (int shift = 0; shift < 8; ++shift) {
        const int g0 = -L - shift;
        int n = 0;
        for (const PairTriple& t : triples) n += (t.l - g0) / 8 - (-t.l - g0) / 8 + 1;
        if ((L - g0) / 8 + 1 > (2 * L + 1 + 7) / 8) continue;                  // no more chunks than needed
        if (best < 0 || n < best) { best = n; out->grid0 = g0; }
    }
    out->nchunks = (L - out->grid0) / 8 + 1;
    for (int v = kVariants - 1; v >= 0; --v)
        if (L <= kVariantL[v]) out->variant = v;
    const size_t most = 4 * kVariantKS[out->variant];                          // output degrees of a pair
    std::vector<double> tile_cost;
    std::vector<int2> coefmap;
    size_t coef = 0, lds = 0;
    for (size_t from = 0, to; from < order.size(); from = to) {
        to = from + 1;
        while (to < order.size() && to - from < most && std::equal(order[to].begin(), order[to].begin() + 3, order[from].begin())) ++to;
        BackPair p{};
        p.l1 = order[from][0]; p.l2 = order[from][1];
        p.tau1 = t_F[p.l1]; p.tau2 = t_F[p.l2];
        p.nl = (int)(to - from);
        p.nks = (p.nl + 3) / 4;
        p.nt = (2 * p.l2 + 1 + 15) / 16;
        // Whole rows t1 in a tile, or sixteen columns wherever they begin, where that makes fewer tiles (tau2 = 12: nine for 144
        // channels, not twelve); the latter repeat their t2 after tau2 / gcd(16, tau2) tiles.
        const int C = p.tau1 * p.tau2, whole = std::min(std::min(kBackMaxTau / p.tau2, p.tau1), kBackMaxRows);
        p.ncol = whole * p.tau2;
        p.tstep = 1;
        if ((C + 15) / 16 < (p.tau1 + whole - 1) / whole && (14 + p.tau2) / p.tau2 + 1 <= kBackMaxRows) {
            p.ncol = kBackMaxTau;
            p.tstep = p.tau2 / std::gcd(16, p.tau2);
        }
        p.ntiles = (C + p.ncol - 1) / p.ncol;
        for (int t = 0; t < p.ntiles; ++t)
            p.nrows = std::max(p.nrows, (std::min(C, (t + 1) * p.ncol) - 1) / p.tau2 - t * p.ncol / p.tau2 + 1);
        p.inv_tau2 = (65536 + p.tau2 - 1) / p.tau2;
        p.inv_M1 = ((1 << 20) + 2 * p.l1) / (2 * p.l1 + 1);
        p.inv_M2 = ((1 << 20) + 2 * p.l2) / (2 * p.l2 + 1);
        const int lm = -order[from][3];
        p.c0 = (-lm - out->grid0) / 8;
        p.nch = (lm - out->grid0) / 8 - p.c0 + 1;
        p.offF1 = cumF[p.l1]; p.offF2 = cumF[p.l2];
        p.coef = (int)coef;
        for (int q = 0; q < p.nl; ++q) {
            const PairTriple& t = triples[order[from + q][4]];
            p.l[q] = t.l;
            p.l8[q >> 2] |= (unsigned)t.l << (8 * (q & 3));
            p.cg[q] = t.cg;
            p.offFF[q] = t.offFF;
            if (p.offFF[q] == 0) p.ends |= 1;
            if (p.offFF[q] + p.tau1 * p.tau2 * (2 * p.l[q] + 1) == nFF) p.ends |= 2;
        }
        // cycles of a tile: matrix instructions of H, the vector half, making (or fetching and turning) G
        double cost = 3000;
        for (int x = 0; x < 8 * p.nch; ++x) {
            const int M = out->grid0 + 8 * p.c0 + x;
            int n = 0, tiles = 0;
            for (int q = 0; q < p.nl; ++q) n += std::abs(M) <= p.l[q];
            for (int rt = 0; rt < p.nt && n > 0; ++rt) {
                const int lo = std::max(-p.l2, M - p.l1), hi = std::min(p.l2, M + p.l1);
                if (lo <= -p.l2 + 16 * rt + 15 && hi >= -p.l2 + 16 * rt) tiles |= 1 << rt;
            }
            const int nk = tiles ? (n + 3) / 4 : 0;
            p.steps[x >> 3] |= nk << (4 * (x & 7));
            p.tiles[x >> 3] |= tiles << (4 * (x & 7));
            p.degs[x >> 3] = std::max(p.degs[x >> 3], n);
            const int entries = std::min(p.l2, M + p.l1) - std::max(-p.l2, M - p.l1) + 1;
            if (n > 0) out->macs += (double)C * n * entries;
            out->blocks += (double)p.ntiles * __builtin_popcount(tiles);
            if (nk > 0) coefmap.push_back(make_int2((int)out->pairs.size(), x));
            cost += 60 + __builtin_popcount(tiles) * (64. * nk + 110.);
        }
        out->tiles += p.ntiles;
        for (int c = 0; c < p.nch; ++c) cost += ((p.degs[c] + 3) / 4) * 4 * 220.;
        tile_cost.push_back(cost);
        coef += (size_t)8 * p.nch * p.nks * p.nt * 64;
        p.nbuf = p.ntiles > p.tstep ? 2 : 1;
        lds = std::max(lds, (size_t)back_lds_floats(p.nch, p.nt, p.nrows, p.nbuf));
        out->pairs.push_back(p);
    }
    CGNET_REQUIRE(coef < (1u << 30), CGNET_ERR_UNSUPPORTED, "packed coefficients of the backward exceed 2^30 floats");
    out->coef_floats = coef + 64 * 4 * 3;          // a chunk's last reads may run past its own groups
    out->ncoefmap = (int)coefmap.size();
    out->lds = 4 * lds * kBackWaves;
    // levels: pieces of at most 1 / n of a sample's work, for batches that make about 5120 units of them: enough waves that the longest
    // is a small part of the call
    double all = 0;
    for (size_t k = 0; k < tile_cost.size(); ++k) all += tile_cost[k] * out->pairs[k].ntiles;
    std::vector<int> cum_rows(L + 2, 0);
    for (int l = 0; l <= L; ++l) cum_rows[l + 1] = cum_rows[l] + t_F[l];
    std::vector<std::vector<int>> combine;
    for (const int n : {64, 256, 1 << 30}) {
        BackLevel lv;
        lv.least_B = n == 1 << 30 ? 1 : (5120 + n - 1) / n;
        const double target = n == 1 << 30 ? 0. : all / n;
        std::vector<std::pair<double, BackUnit>> units;
        std::vector<int4> shares;                                   // (row of a degree, where a share of it lies, which, tiles of back_share)
        int at = 0;
        for (size_t k = 0; k < out->pairs.size(); ++k) {
            const BackPair& p = out->pairs[k];
            const int M1 = 2 * p.l1 + 1, M2 = 2 * p.l2 + 1;
            for (int phase = 0; phase < std::min(p.tstep, p.ntiles); ++phase) {
                const int nt = (p.ntiles - phase + p.tstep - 1) / p.tstep;
                const int pieces = target > 0. ? std::max(1, (int)std::min((double)nt, std::ceil(nt * tile_cost[k] / target))) : nt;
                for (int i = 0; i < pieces; ++i) {
                    const int t0 = nt * i / pieces, n = nt * (i + 1) / pieces - t0;
                    BackUnit u{(int)k, phase + t0 * p.tstep, n, at, 0};
                    for (int t = 0; t < n; ++t) {
                        const int c0 = (u.tile0 + t * p.tstep) * p.ncol, c1 = std::min(p.tau1 * p.tau2, c0 + p.ncol);
                        for (int r = c0 / p.tau2; r <= (c1 - 1) / p.tau2; ++r)
                            shares.push_back(make_int4(cum_rows[p.l1] + r, at + (t * p.nrows + r - c0 / p.tau2) * M1, 2 * (int)k,
                                                       (u.tile0 + t * p.tstep) | 1 << 16));
                    }
                    at += n * p.nrows * M1;
                    u.p2off = at;
                    for (int r = 0; r < p.tau2; ++r)
                        shares.push_back(make_int4(cum_rows[p.l2] + r, at + r * M2, 2 * (int)k + 1, u.tile0 | n << 16));
                    at += p.tau2 * M2;
                    units.push_back({tile_cost[k] * n, u});
                }
            }
        }
        std::stable_sort(units.begin(), units.end(), [](const auto& x, const auto& y) { return x.first > y.first; });
        for (const auto& x : units) lv.units.push_back(x.second);
        lv.P = at;
        // meta of cg_backward_rows_kernel
        std::vector<int> meta(cumF.begin(), cumF.end());
        meta.insert(meta.end(), cum_rows.begin(), cum_rows.end());
        const size_t head = meta.size(), nrows = cum_rows[L + 1];
        meta.resize(head + nrows + 1 + 3 * shares.size());
        int* begin = meta.data() + head;                            // (counted one place on, then summed)
        for (const int4& x : shares) ++begin[x.x + 1];
        for (size_t r = 0; r < nrows; ++r) begin[r + 1] += begin[r];
        std::vector<int> next(begin, begin + nrows);
        int *offset = begin + nrows + 1, *which = offset + shares.size();
        for (const int4& x : shares) {
            const int to = next[x.x]++;
            offset[to] = x.y;
            which[2 * to] = x.z;
            which[2 * to + 1] = x.w;
        }
        bool finest = true;
        for (const BackUnit& u : lv.units) finest &= u.ntiles == 1;
        out->levels.push_back(lv);
        combine.push_back(meta);
        if (finest) {
            out->levels.back().least_B = 1;
            break;
        }
    }
    // everything in one allocation, filled by one copy
    size_t bytes = 0;
    auto place = [&](size_t n) { const size_t at = bytes; bytes += align_up(n, 256); return at; };
    const size_t at_pairs = place(sizeof(BackPair) * out->pairs.size()), at_map = place(sizeof(int2) * coefmap.size());
    std::vector<size_t> at_units, at_meta;
    for (size_t k = 0; k < out->levels.size(); ++k) {
        at_units.push_back(place(sizeof(BackUnit) * out->levels[k].units.size()));
        at_meta.push_back(place(sizeof(int) * combine[k].size()));
    }
    const std::unique_ptr<unsigned char[]> host(new unsigned char[bytes]());
    memcpy(host.get() + at_pairs, out->pairs.data(), sizeof(BackPair) * out->pairs.size());
    memcpy(host.get() + at_map, coefmap.data(), sizeof(int2) * coefmap.size());
    for (size_t k = 0; k < out->levels.size(); ++k) {
        memcpy(host.get() + at_units[k], out->levels[k].units.data(), sizeof(BackUnit) * out->levels[k].units.size());
        memcpy(host.get() + at_meta[k], combine[k].data(), sizeof(int) * combine[k].size());
    }
    CGNET_HIP(hipMalloc((void**)&out->d_tables, bytes));
    CGNET_HIP(hipMemcpy(out->d_tables, host.get(), bytes, hipMemcpyHostToDevice));
    out->d_pairs = reinterpret_cast<BackPair*>(out->d_tables + at_pairs);
    out->d_coefmap = reinterpret_cast<int2*>(out->d_tables + at_map);
    for (size_t k = 0; k < out->levels.size(); ++k) {
        out->levels[k].d_units = reinterpret_cast<BackUnit*>(out->d_tables + at_units[k]);
        out->levels[k].d_combine = reinterpret_cast<int*>(out->d_tables + at_meta[k]);
    }
    return raise_dynamic_lds(variant_kernel(out->variant, 0), out->lds);
}

int launch_pack_coef_back(const BackSet& set, const float* d_CG, float* d_coef, hipStream_t s) {
    CGNET_LAUNCH(pack_coef_back_kernel, dim3((unsigned)set.ncoefmap), dim3(256), 0, s, d_CG, set.d_pairs, set.d_coefmap, set.grid0,
                 d_coef);
    CGNET_HIP(hipGetLastError());
    return CGNET_OK;
}

int launch_back_memory(const BackSet& set, const BackLevel& lv, const float* d_F, const float* d_gFF, const float* d_coef,
                       float* d_part, float* d_gF, int L, int nF, int nFF, int B, hipStream_t s) {
    BackArgs a{};
    a.F = (const float2*)d_F; a.gFF = (const float2*)d_gFF;
    a.coef = d_coef; a.part = (float2*)d_part;
    a.nF = nF; a.nFF = nFF; a.B = B;
    BackTerms t{};
    t.F = a.F; t.gFF = a.gFF; t.nFF = nFF; t.coef = d_coef;
    return launch_back(set, lv, kBackMemory, a, t, d_gF, L, s);
}

// ---- layer source --------------------------------------------------------------------------------
void free_back_link(BackLink* link) {
    if (link->d_tables) (void)hipFree(link->d_tables);
    *link = BackLink();
}

int build_back_link(const cgnet_cg_plan* p, const cgnet_wmm_plan* w, BackLink* link) {
    free_back_link(link);
    CGNET_REQUIRE(wmm_plan_degrees(w) == p->L + 1, CGNET_ERR_ARG, "the two plans have different lmax");
    std::vector<WmmDegInfo> info(p->L + 1);
    for (int l = 0; l <= p->L; ++l) {
        if (int rc = wmm_plan_degree(w, l, &info[l])) return rc;
        CGNET_REQUIRE(info[l].K == p->t_FF[l], CGNET_ERR_ARG,
                      "degree %d: the mixing plan has %d mid channels, the product %d", l, info[l].K, p->t_FF[l]);
    }
    const BackSet& set = p->back;
    CGNET_REQUIRE(set.ok(), CGNET_ERR_UNSUPPORTED,
                  "the fused backward needs lmax <= %d and at most %d channels in every input degree", kBackMaxL, kBackMaxTau);
    CGNET_REQUIRE(wmm_gradff_operand_ok(w), CGNET_ERR_UNSUPPORTED, "the fused backward needs t_O <= 16 in every degree");
    link->nO = info[p->L].cumO + info[p->L].tO * (2 * p->L + 1);
    int most = 0;
    std::vector<int2> degs(p->L + 1);
    for (int l = 0; l <= p->L; ++l) {
        degs[l] = make_int2(info[l].cumO, info[l].tO);
        most = std::max(most, info[l].tO);
    }
    const bool split = split_taken(p->L, [&](int l) { return info[l].tO; });
    link->source = split ? kBackSplit : std::max(1, (most + 3) / 4);
    link->lanes = split ? 16 * ((most + 3) / 4) : 64;
    const int places = set.nchunks * (p->L + 1);
    link->go_degree = split ? set.nchunks * kBackOperand : 128 * link->source;
    link->go_flags = split ? places * kBackOperand + set.nchunks * kBackScales : places * 128 * link->source;
    link->go_floats = (int)align_up(link->go_flags + places, 64);
    std::vector<int> reach((p->L + 1) * (p->L + 1), -1);
    for (const BackPair& b : set.pairs)
        for (int q = 0; q < b.nl; ++q) {
            int &r1 = reach[b.l1 * (p->L + 1) + b.l[q]], &r2 = reach[b.l2 * (p->L + 1) + b.l[q]];
            r1 = std::max(r1, b.l2);
            r2 = std::max(r2, b.l1);
        }
    std::vector<BackGenPair> gps(set.pairs.size());
    std::vector<BackGenW> gens;
    size_t at = 0;
    for (size_t k = 0; k < set.pairs.size(); ++k) {
        const BackPair& b = set.pairs[k];
        BackGenPair& g = gps[k];
        g = BackGenPair{};
        g.w = (int)at;
        g.wtile = split ? b.nl * kBackOperand : b.nks * 512 * link->source;
        for (int q = 0; q < b.nl; ++q) {
            const int l = b.l[q];
            BackGenW e{};
            e.chan0 = (b.offFF[q] - p->cumFF[l]) / (2 * l + 1);
            e.nch = b.tau1 * b.tau2;
            e.tO = info[l].tO; e.cumW = info[l].cumW; e.K = info[l].K; e.cumT = info[l].cumT;
            e.source = link->source;
            e.at = (int)at + (split ? kBackOperand * q : (q / 4) * 512 * link->source + 256 * (q / 2 % 2) + 2 * (q & 1));
            e.ncol = b.ncol;
            e.ntiles = b.ntiles;
            e.wtile = g.wtile;
            gens.push_back(e);
        }
        at += (size_t)g.wtile * b.ntiles;
        CGNET_REQUIRE(at < (1u << 30), CGNET_ERR_UNSUPPORTED, "packed weights of the fused backward exceed 2^30 floats");
    }
    link->w_floats = at + 2 * kBackOperand;         // fetches run ahead of a tile's degrees
    link->ngens = (int)gens.size();
    size_t bytes = 0;
    auto place = [&](size_t n) { const size_t o = bytes; bytes += align_up(n, 256); return o; };
    const size_t at_gp = place(sizeof(BackGenPair) * gps.size()), at_gd = place(sizeof(int2) * degs.size());
    const size_t at_gw = place(sizeof(BackGenW) * gens.size()), at_reach = place(sizeof(int) * reach.size());
    const std::unique_ptr<unsigned char[]> host(new unsigned char[bytes]());
    memcpy(host.get() + at_gp, gps.data(), sizeof(BackGenPair) * gps.size());
    memcpy(host.get() + at_gd, degs.data(), sizeof(int2) * degs.size());
    memcpy(host.get() + at_gw, gens.data(), sizeof(BackGenW) * gens.size());
    memcpy(host.get() + at_reach, reach.data(), sizeof(int) * reach.size());
    CGNET_HIP(hipMalloc((void**)&link->d_tables, bytes));
    if (hipMemcpy(link->d_tables, host.get(), bytes, hipMemcpyHostToDevice) != hipSuccess) {
        free_back_link(link);
        set_error("copying the tables of the fused backward failed");
        return CGNET_ERR_HIP;
    }
    link->d_gp = reinterpret_cast<BackGenPair*>(link->d_tables + at_gp);
    link->d_degs = reinterpret_cast<int2*>(link->d_tables + at_gd);
    link->d_reach = reinterpret_cast<int*>(link->d_tables + at_reach);
    link->d_gens = reinterpret_cast<BackGenW*>(link->d_tables + at_gw);
    link->ndeg = p->L + 1;
    link->most_B = p->bwd_hybrid ? back_most_batch(set, p->L, p->nFF, (int)p->bwd_utasks.size(), kBackRuleLayer) : INT32_MAX;
    if (int rc = raise_dynamic_lds(variant_kernel(set.variant, link->source), set.lds)) {
        free_back_link(link);
        return rc;
    }
    link->ok = true;
    return CGNET_OK;
}

int launch_pack_w_back(const BackLink& link, const float* d_W, const float* d_stds, float eps, float* d_Wp, hipStream_t s) {
    CGNET_LAUNCH(pack_w_back_kernel, dim3((unsigned)link.ngens), dim3(256), 0, s, (const float2*)d_W, d_stds, eps, link.d_gens, d_Wp);
    CGNET_HIP(hipGetLastError());
    return CGNET_OK;
}

int launch_back_layer(const BackSet& set, const BackLink& link, const BackLevel& lv, const float* d_F, const float* d_gO,
                      const float* d_Wp, const float* d_coef, float* d_Go, float* d_part, float* d_gF, int L, int nF, int B,
                      hipStream_t s) {
    CGNET_REQUIRE(B <= 65535, CGNET_ERR_UNSUPPORTED, "B=%d above 65535", B);
    const bool split = link.source == kBackSplit;
    const int places = set.nchunks * link.ndeg;
    if (split)
        CGNET_LAUNCH(pack_go_back_split_kernel, dim3((unsigned)set.nchunks, (unsigned)B), dim3(64 * kPackGoWaves), 0, s, (const float2*)d_gO,
                     link.d_degs, d_Go, link.ndeg, set.grid0, link.nO, link.go_floats);
    else
        CGNET_LAUNCH(pack_go_back_kernel, dim3((unsigned)(set.nchunks * link.ndeg), (unsigned)B), dim3(64), 0, s, (const float2*)d_gO,
                     link.d_degs, d_Go, link.ndeg, link.source, set.grid0, link.nO, link.go_floats);
    CGNET_HIP(hipGetLastError());
    BackArgs a{};
    a.F = (const float2*)d_F; a.Go = d_Go; a.W = d_Wp; a.gp = link.d_gp;
    a.coef = d_coef; a.part = (float2*)d_part;
    a.nF = nF; a.nGo = link.go_floats; a.go_degree = link.go_degree; a.go_chunk = split ? kBackOperand : link.ndeg * link.go_degree;
    a.go_scales = kBackOperand * places; a.lanes = link.lanes; a.B = B;
    BackTerms t{};
    t.gO = (const float2*)d_gO; t.degs = link.d_degs; t.reach = link.d_reach; t.nO = link.nO; t.ndeg = link.ndeg;
    t.odd = reinterpret_cast<const int*>(d_Go) + link.go_flags; t.nodd = places; t.nGo = link.go_floats;
    return launch_back(set, lv, link.source, a, t, d_gF, L, s);
}

}  // namespace cgnet
