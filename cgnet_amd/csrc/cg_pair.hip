// Clebsch-Gordan product organised by pairs of input degrees, for gfx950.
//
// For a pair (l1, l2) every output degree l contracts the same products of fragment entries with its own
// coefficients:
//     FF_l[t1, t2, m] = sum_m2 C_l[m][m2] P[t1, t2][m - m2, m2],     P[t1, t2][m1, m2] = F1[t1][m1] F2[t2][m2].
// A unit takes four output degrees of a pair at once.  A lane is one channel (t1, t2) of one sample -- a wave is filled
// with several samples where a pair has few channels -- and forms P on the vector ALUs (four instructions); all lanes
// then need the same four coefficients, which is what v_mfma_f32_4x4x1_16b_f32 does with a broadcast left operand:
// rows = the four degrees, columns = the 64 lanes, so an instruction of eight cycles is four multiply-adds per lane,
// and its coefficients cost one 4-byte read per lane and four steps.  (Measured on this GPU: a plain fp32 vector
// multiply-add takes 2.3 cycles of a SIMD, one with a scalar or a DPP operand 4.3, the matrix instruction 8.5;
// coefficients through scalar registers or row broadcasts therefore cost twice as much.)
#include <algorithm>
#include <array>
#include <cstring>
#include <map>

#include "cg_pair.h"
#include "internal.h"

namespace cgnet {
namespace {

constexpr int kPairThreads = 64 * kPairWaves;
constexpr size_t kPairMaxLds = 160 * 1024;
constexpr size_t kPairMaxCoef = 32 * 1024;      // coefficients of a unit kept in LDS; beyond that every wave fetches an item's
                                                // as it comes to it (degrees above 23 only)
constexpr int kPairPad = 4;                     // zeros behind every staged row: the steps of an item that lie past a row's end
                                                // read them

typedef float v2f __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(3))) v2f* lds_v2_p;
typedef const __attribute__((address_space(3))) float* lds_f_p;
typedef const __attribute__((address_space(4))) int* scalar_i_p;           // uniform loads go through the scalar cache

__device__ __forceinline__ unsigned lds_address(const void* p) {
    return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ v2f lds_read(unsigned a) { return *(lds_v2_p)(uintptr_t)a; }
__device__ __forceinline__ float lds_read1(unsigned a) { return *(lds_f_p)(uintptr_t)a; }

// LDS before the coefficients: two buffers of (zeros | S x rows of degree l1 | S x channels of degree l2, each with zeros
// behind it), then one row of zeros for lanes without a channel
__host__ __device__ inline int pair_slab_floats(const FwdPair& u, int S) {
    return 2 * (kPairPad + S * (u.rows * (2 * u.l1 + 1 + kPairPad) + u.nt2 * (2 * u.l2 + 1 + kPairPad)));
}
__host__ __device__ inline size_t pair_front_bytes(const FwdPair& u, int S) {
    return ((((size_t)4 * pair_slab_floats(u, S) + 15) & ~(size_t)15) * 2 + 8 * (2 * u.l1 + 1 + 2 * kPairPad) + 15) & ~(size_t)15;
}

// Starts the copy of `rows` rows of M complex entries per sample (S samples, `stride` floats apart) to LDS rows of
// M + kPairPad entries behind dst: a row at a time, dealt to the waves.
__device__ __forceinline__ void stage_rows(const float* __restrict__ src, size_t stride, int rows, int M, int S, float* dst,
                                           int wave, int lane) {
    const int pitch = 2 * (M + kPairPad);
    int t = wave;
    for (int s = 0; s < S; ++s, t -= rows) {
        for (; t < rows; t += kPairWaves)
            for (int x = 0; x < 2 * M; x += 64)
                if (x + lane < 2 * M)
                    __builtin_amdgcn_global_load_lds(src + (size_t)s * stride + t * 2 * M + x + lane,
                                                     (lds_void_ptr)(dst + (s * rows + t) * pitch + x), 4, 0, 0);
    }
}

__device__ __forceinline__ v2f cmul(v2f f, v2f g) { return (v2f){fmaf(f.x, g.x, -f.y * g.y), fmaf(f.x, g.y, f.y * g.x)}; }

// acc[k] += (coefficient k of step ABID) * p: rows of the left operand's block ABID are broadcast to all sixteen blocks
template <int ABID>
__device__ __forceinline__ void step4(f32x4& re, f32x4& im, float c, v2f p) {
    re = __builtin_amdgcn_mfma_f32_4x4x1f32(c, p.x, re, 4, ABID, 0);
    im = __builtin_amdgcn_mfma_f32_4x4x1f32(c, p.y, im, 4, ABID, 0);
}

// N steps (two or four) of an item.  pf, pg: LDS addresses of F1[m - m2] and F2[m2] of the first; fn = F1[m + 1 - m2].
template <int N>
__device__ __forceinline__ void item_steps(unsigned& pf, unsigned& pg, unsigned& pc, unsigned wofs, v2f& fn, f32x4& re0, f32x4& im0,
                                           f32x4& re1, f32x4& im1) {
    v2f f[N], g[N];
    pf -= 8 * (N - 1);
#pragma unroll
    for (int u = 0; u < N; ++u) {
        f[u] = lds_read(pf + 8 * (N - 1 - u));
        g[u] = lds_read(pg + 8 * u);
    }
    const float w0 = lds_read1(pc), w1 = lds_read1(pc + wofs);
    step4<0>(re0, im0, w0, cmul(f[0], g[0]));
    step4<0>(re1, im1, w1, cmul(fn, g[0]));
    step4<1>(re0, im0, w0, cmul(f[1], g[1]));
    step4<1>(re1, im1, w1, cmul(f[0], g[1]));
    if constexpr (N == 4) {
        step4<2>(re0, im0, w0, cmul(f[2], g[2]));
        step4<2>(re1, im1, w1, cmul(f[1], g[2]));
        step4<3>(re0, im0, w0, cmul(f[3], g[3]));
        step4<3>(re1, im1, w1, cmul(f[2], g[3]));
    }
    fn = f[N - 1];
    pc += 2 * N * wofs;
    pf -= 8;
    pg += 8 * N;
}

// this wave's LDS accesses are complete, then the group's barrier; copies and stores stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// both sums run over the same rounded |z| in double: the variance formed from them is then free of cancellation between
// inconsistently rounded terms
__device__ __forceinline__ void add_modulus(float re, float im, double& s1, double& s2) {
    const double d = (double)__builtin_amdgcn_sqrtf(fmaf(re, re, im * im));
    s1 += d;
    s2 = fma(d, d, s2);
}

// LDS: staged fragments (pair_slab_floats) | a row of zeros | coefficients, per item and step the four degrees' values for m,
// then for m + 1 | tile, per output degree [64 slots][2l+1] complex.
//
// What the kernel is short of, beside the HBM writes, is instruction issue, and above all scalar issue (the scalar unit
// serves the four SIMDs of a compute unit in turn): items are described by the plan, the staged rows are padded with
// zeros so that an item is a plain loop over blocks of four steps, and nothing is decided per step.  What is left is
// mostly latency: the fetch of the coefficients when a work-group starts, and the two barriers of a stage.
// Measured (with statistics, against the vector-ALU kernel cg_forward_kernel that these shapes ran before): lmax 10, 12 .. 3
// channels, B = 100 (63 MB of product): 119 -> 54 us; lmax 11, 5 channels, B = 32 (43 MB): 69 -> 40 us; lmax 20, 1 channel,
// B = 32: 252 -> 98 us; lmax 13, minimum-spanning-tree triples, 16 .. 4 channels, B = 27: 49 -> 34 us.
// LOCAL: the units' coefficients do not fit the LDS (FwdPair::cg_local); a variant of its own because a global load inside
// the item loop makes the compiler wait there for every copy in flight.
template <bool STATS, bool LOCAL>
__global__ void __launch_bounds__(kPairThreads, 5)
cg_forward_pair_kernel(const float2* __restrict__ F, float2* __restrict__ FF, const float* __restrict__ CG,
                  const FwdPair* __restrict__ units, const FwdItem* __restrict__ items, int nF, int nFF, int B,
                  int samples_per_group, double* __restrict__ stats_part, int sumT) {
    extern __shared__ __align__(16) unsigned char smem[];
    const UnitPart up = part_major((B + samples_per_group - 1) / samples_per_group);
    const FwdPair& u = units[up.unit];
    const int group = up.part;
    const int l1 = u.l1, l2 = u.l2, nl = u.nl, nc = u.nc;
    const int S = min(u.S, samples_per_group);
    const int M1 = 2 * l1 + 1, M2 = 2 * l2 + 1;
    const int slab = pair_slab_floats(u, S);
    const int front = (int)pair_front_bytes(u, S), second = (4 * slab + 15) & ~15;
    float* frag = reinterpret_cast<float*>(smem);
    float* cgs = reinterpret_cast<float*>(smem + front);
    float* tile = reinterpret_cast<float*>(smem + front + u.cgbytes);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // lane -> (sample of the stage, channel)
    const int ls = min(lane / nc, S - 1);
    const int lc = min(lane - ls * nc, nc - 1);
    const int t1 = (u.c0 + lc) / u.tau2, t2 = (u.c0 + lc) - t1 * u.tau2;
    const int part2 = kPairPad + S * u.rows * (M1 + kPairPad);          // complex index of the first row of degree l2
    const unsigned base = lds_address(smem);
    const unsigned b1 = base + 8u * (unsigned)(kPairPad + (ls * u.rows + t1 - u.r0) * (M1 + kPairPad) + l1);
    const unsigned b2 = base + 8u * (unsigned)(part2 + (ls * u.nt2 + t2 - u.q0) * (M2 + kPairPad) + l2);
    const unsigned bz = base + 2u * (unsigned)second + 8u * (unsigned)(kPairPad + l1);
    for (int e = tid; e < front >> 4; e += kPairThreads)
        reinterpret_cast<float4*>(smem)[e] = make_float4(0.f, 0.f, 0.f, 0.f);

    unsigned out[kPairNL];                                             // per output degree: where the lane's results for m = 0 go
    {
        unsigned t0 = lds_address(tile);
#pragma unroll
        for (int k = 0; k < kPairNL; ++k) {
            const int M = 2 * u.l[k] + 1;
            out[k] = t0 + 8u * (unsigned)(lane * M + u.l[k]);
            t0 += 512u * (unsigned)M;
        }
    }
    double s1[kPairNL], s2[kPairNL];
#pragma unroll
    for (int k = 0; k < kPairNL; ++k) s1[k] = s2[k] = 0.;

    const int first = group * samples_per_group;
    const int last = min(B, first + samples_per_group);
    auto issue = [&](int b, int par) {
        const int ns = min(S, last - b);
        const float* Fb = reinterpret_cast<const float*>(F + (size_t)b * nF);
        stage_rows(Fb + 2 * u.offF1, 2 * (size_t)nF, u.rows, M1, ns, frag + par * (second >> 2) + 2 * kPairPad, wave, lane);
        stage_rows(Fb + 2 * u.offF2, 2 * (size_t)nF, u.nt2, M2, ns, frag + par * (second >> 2) + 2 * part2, wave, lane);
    };
    __syncthreads();                                                   // the zeros precede every copy
    issue(first, 0);

    // Coefficients: a wave fetches those of its own items, lane = (one of eight steps, m or m + 1, degree), four fetches in
    // flight at a time.
    const int turn = (wave + (int)blockIdx.x) & (kPairWaves - 1);      // which SIMD gets which share varies over the groups
    const scalar_i_p wi = (scalar_i_p)(uintptr_t)(items + u.item0 + u.wbeg[turn]);
    const int nmine = u.wbeg[turn + 1] - u.wbeg[turn], local = u.cg_local;
    const int fk = lane & 3, fwhich = (lane >> 2) & 1, fl = u.l[fk], fcg = u.cg[fk];
    auto fetch = [&](int m8, int lo, int x) -> float {
        const int mm = (m8 >> 3) + fwhich, m2 = lo + x, m1 = mm - m2;
        return mm >= -fl && mm <= fl && m1 >= -l1 && m1 <= l1 && m2 <= l2 ? CG[fcg + (mm + fl) * M2 + m2 + l2] : 0.f;
    };
    auto steps_of = [](int shape) { return 4 * (shape & 255) + 2 * ((shape >> 8) & 1); };
    if (!LOCAL) {
        int j = 0, x0 = 0;
        while (j < nmine) {
            float v[4];
            int to[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                to[q] = -1;
                if (j < nmine) {
                    const scalar_i_p it = wi + 8 * j;
                    const int steps = steps_of(it[4]), x = x0 + (lane >> 3);
                    if (x < steps && fk < nl) {
                        to[q] = (it[3] >> 2) + (2 * x + fwhich) * nl + fk;
                        v[q] = fetch(it[0], it[2] >> 3, x);
                    }
                    x0 += 8;
                    if (x0 >= steps) { x0 = 0; ++j; }
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (to[q] >= 0) cgs[to[q]] = v[q];
        }
    }
    // lane -> (step of a block of four, degree); rows past the unit's degrees read whatever follows, nobody uses their sums
    const unsigned wofs = 4u * (unsigned)nl;
    const unsigned pc0 = lds_address(cgs) + 2u * wofs * (unsigned)((lane & 15) >> 2) + 4u * (unsigned)(lane & 3);
    // the degree this wave copies out (waves beyond the unit's degrees have none)
    const int kout = wave < nl ? wave : -1;
    const int nout = kout >= 0 ? nc * (2 * u.l[kout] + 1) : 0;         // entries of one sample
    int tile_out = 0;                                                  // its first entry in the tile
    for (int k = 0; k < kout; ++k) tile_out += 64 * (2 * u.l[k] + 1);
    float2* const dst0 = FF + (kout >= 0 ? u.offFF[kout] : 0);
    const int nstores = max(1, nout >> 7);                             // at least so many stores follow a stage's copies
    int par = 0;
    for (int b = first; b < last; b += S, par ^= 1) {
        // this stage's fragments have landed (the stores of the previous stage, issued after their copies, stay in flight)
        if (b == first || kout < 0) dma_wait();
        else wait_vmcnt(min(nstores, 28));
        lds_barrier();                         // ... for every wave; the previous tile has been copied out
        if (b + S < last) issue(b + S, par ^ 1);
        const int ns = min(S, last - b);
        const bool valid = lane < ns * nc;
        const unsigned a1 = valid ? b1 + (unsigned)(par * second) : bz, a2 = valid ? b2 + (unsigned)(par * second) : bz;
        for (int j = 0; j < nmine; ++j) {
            const scalar_i_p it = wi + 8 * j;
            const int m8 = it[0], shape = it[4];
            int place = it[3];
            if (LOCAL) {                                               // this wave's own buffer, filled for every item
                place = wave * local;
                for (int x = lane >> 3; x < steps_of(shape); x += 8)
                    if (fk < nl) cgs[(place >> 2) + (2 * x + fwhich) * nl + fk] = fetch(m8, it[2] >> 3, x);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
            unsigned pf = a1 + (unsigned)it[1], pg = a2 + (unsigned)it[2], pc = pc0 + (unsigned)place;
            v2f fn = lds_read(pf + 8);
            f32x4 re0 = {0.f, 0.f, 0.f, 0.f}, im0 = re0, re1 = re0, im1 = re0;
            for (int n4 = shape & 255; n4 > 0; --n4) item_steps<4>(pf, pg, pc, wofs, fn, re0, im0, re1, im1);
            if (shape & 256) item_steps<2>(pf, pg, pc, wofs, fn, re0, im0, re1, im1);
            // results -> tile (degrees without the value hold zero sums)
            const int nb = (shape >> 16) & 255, part = shape >> 24;
            typedef __attribute__((address_space(3))) v2f* lds_w_p;
#pragma unroll
            for (int k = 0; k < kPairNL; ++k) {
                const lds_w_p o = (lds_w_p)(uintptr_t)(out[k] + (unsigned)m8);
                if (k < nb) {
                    o[0] = (v2f){re0[k], im0[k]};
                    o[1] = (v2f){re1[k], im1[k]};
                    if (STATS) {
                        add_modulus(re0[k], im0[k], s1[k], s2[k]);
                        add_modulus(re1[k], im1[k], s1[k], s2[k]);
                    }
                } else {
                    if (k == nb && part) {
                        const v2f z = part == 1 ? (v2f){re0[k], im0[k]} : (v2f){re1[k], im1[k]};
                        o[part - 1] = z;
                        if (STATS) add_modulus(z.x, z.y, s1[k], s2[k]);
                    }
                    break;
                }
            }
        }
        lds_barrier();
        // tile -> FF, one degree per wave: per sample one contiguous run, 16 bytes per lane (its start is 8-byte aligned)
        const float2* src = reinterpret_cast<const float2*>(tile) + tile_out;
        float2* dst = dst0 + (size_t)b * nFF;
        const int npair = nout >> 1;
        if (npair >= 48 || ns == 1) {
            for (int s = 0; s < ns; ++s, src += nout, dst += nFF) {
                const float2* x = src + 2 * lane;
                float2* y = dst + 2 * lane;
                int left = npair - lane;
#pragma unroll 4
                for (int it = npair >> 6; it > 0; --it, x += 128, y += 128, left -= 64)
                    stream_store16(y, x[0].x, x[0].y, x[1].x, x[1].y);
                if (left > 0) stream_store16(y, x[0].x, x[0].y, x[1].x, x[1].y);
                if ((nout & 1) && lane == 0) dst[nout - 1] = src[nout - 1];
            }
        } else if (nout > 0) {
            const int nw = (nout + 1) >> 1;                            // 16-byte pieces of a sample, the last may be half
            const float inv = 1.f / (float)nw;
            for (int j = lane; j < ns * nw; j += 64) {
                const int s = (int)(((float)j + 0.5f) * inv), e = 2 * (j - s * nw);
                const float2* x = src + s * nout + e;
                float2* y = dst + (size_t)s * nFF + e;
                if (e + 1 < nout) stream_store16(y, x[0].x, x[0].y, x[1].x, x[1].y);
                else *y = *x;
            }
        }
    }
    if (STATS) {
        // the waves hold partial sums of the same channels (each over its own m), lanes nc apart those of different
        // samples: added in wave order, then sample order
        double2* red = reinterpret_cast<double2*>(smem);               // [degree][wave][lane]
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPairNL; ++k)
            if (k < nl) red[(k * kPairWaves + wave) * 64 + lane] = make_double2(s1[k], s2[k]);
        __syncthreads();
        for (int j = tid; j < nl * nc; j += kPairThreads) {
            const int k = j / nc, c = j - k * nc;
            double a = 0., q = 0.;
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int w = 0; w < kPairWaves; ++w) {
                    const double2 v = red[(k * kPairWaves + w) * 64 + s * nc + c];
                    a += v.x;
                    q += v.y;
                }
            *reinterpret_cast<double2*>(stats_part + ((size_t)group * sumT + u.chan[k] + c) * 2) = make_double2(a, q);
        }
    }
}

}  // namespace

// Samples side by side and channel ranges: a pair of C channels is cut into ranges of at most 64 lanes, and a short range
// takes floor(64 / nc) samples at once.  The cut with the fewest stages per sample (sum of 1 / S), a little dearer per
// range because every range stages the fragments.
static void channel_ranges(int C, int tau2, std::vector<std::pair<int, int>>* out) {
    out->clear();
    if (C <= 64) {
        out->push_back({0, C});
        return;
    }
    if (tau2 > 64) {                        // ranges inside one row t1: few staged channels of degree l2
        const int n = (tau2 + 63) / 64, w = (tau2 + n - 1) / n;
        for (int r = 0; r < C; r += tau2)
            for (int q = 0; q < tau2; q += w) out->push_back({r + q, std::min(w, tau2 - q)});
        return;
    }
    int best = 64;
    double best_cost = -1;
    for (int nc = 16; nc <= 64; ++nc) {
        const int full = C / nc, rest = C % nc;
        const double cost = full * (1. / (64 / nc) + 0.03) + (rest ? 1. / (64 / rest) + 0.03 : 0.);
        if (best_cost < 0 || cost < best_cost - 1e-9) { best_cost = cost; best = nc; }
    }
    for (int c = 0; c < C; c += best) out->push_back({c, std::min(best, C - c)});
}

// Steps (rounded up to pairs) of the item m = 2 p - mh of a pair's m axis -mh .. mh; *lo = its first m2.
static int item_step_count(int l1, int l2, int mh, int p, int* lo) {
    const int m = 2 * p - mh;
    *lo = std::max(-l2, m - l1);
    return 2 * ((std::min(l2, m + (m + 1 <= mh ? 1 : 0) + l1) - *lo + 2) / 2);
}

// LDS bytes of the coefficients of a unit with nl degrees up to mh, all items at once; *most = the largest item's.
static size_t coef_bytes(int l1, int l2, int mh, int nl, size_t* most) {
    size_t bytes = 0;
    *most = 0;
    for (int p = 0, lo; p <= mh; ++p) {
        const size_t b = 8 * (size_t)nl * item_step_count(l1, l2, mh, p, &lo);
        bytes += b;
        *most = std::max(*most, b);
    }
    return bytes + 128;                                           // a read takes four steps, past the last one too
}

// The items of a unit, dealt to the waves (dearest first, always to the wave with the least so far).
static void make_items(FwdPair* u, std::vector<FwdItem>* all) {
    const int mh = u->l[0];
    struct Cand { FwdItem it; int cost, steps; };
    std::vector<Cand> cand;
    cand.reserve(mh + 1);
    for (int p = 0; p <= mh; ++p) {
        const int m = 2 * p - mh;
        const bool two = m + 1 <= mh;
        Cand c;
        int lo;
        c.steps = item_step_count(u->l1, u->l2, mh, p, &lo);
        c.it = FwdItem();
        c.it.m8 = 8 * m;
        c.it.fofs = 8 * (m - lo);
        c.it.gofs = 8 * lo;
        const int half = c.steps / 2;
        int nb = 0, part = 0;
        for (int k = 0; k < u->nl; ++k) {
            const bool in0 = std::abs(m) <= u->l[k], in1 = two && std::abs(m + 1) <= u->l[k];
            if (in0 && in1) ++nb;
            else if (in0 || in1) part = in0 ? 1 : 2;
        }
        c.it.shape = (half / 2) | (half & 1) << 8 | nb << 16 | part << 24;
        c.cost = 60 * c.steps / 4 + 80;
        cand.push_back(c);
    }
    std::stable_sort(cand.begin(), cand.end(), [](const Cand& a, const Cand& b) { return a.cost > b.cost; });
    std::vector<FwdItem> per[kPairWaves];
    long long load[kPairWaves] = {};
    int place = 0;
    for (Cand& c : cand) {
        c.it.place = place;
        place += 8 * u->nl * c.steps;
        int w = 0;
        for (int k = 1; k < kPairWaves; ++k)
            if (load[k] < load[w]) w = k;
        per[w].push_back(c.it);
        load[w] += c.cost;
    }
    u->item0 = (int)all->size();
    u->wbeg[0] = 0;
    for (int w = 0; w < kPairWaves; ++w) {
        all->insert(all->end(), per[w].begin(), per[w].end());
        u->wbeg[w + 1] = u->wbeg[w] + (int)per[w].size();
    }
    size_t most;
    const size_t bytes = coef_bytes(u->l1, u->l2, mh, u->nl, &most);
    u->cg_local = bytes > kPairMaxCoef ? (int)(most + 128) : 0;
    u->cgbytes = (int)align_up(u->cg_local ? kPairWaves * (size_t)u->cg_local : bytes, 16);
}

// The channel range of a unit, the rows and channels it stages, the samples it takes side by side (fewer where their
// fragments would not leave room for the tile).
static void set_channels(FwdPair* u, const std::pair<int, int>& r) {
    u->c0 = r.first; u->nc = r.second; u->S = 64 / r.second;
    u->r0 = r.first / u->tau2;
    u->rows = (r.first + r.second - 1) / u->tau2 - u->r0 + 1;
    u->q0 = u->rows == 1 ? r.first - u->r0 * u->tau2 : 0;
    u->nt2 = u->rows == 1 ? r.second : u->tau2;
    while (u->S > 1 && pair_front_bytes(*u, u->S) > 12 * 1024) --u->S;
}

int build_fwd_pairs(const std::vector<PairTriple>& triples, const std::vector<int>& t_F, const std::vector<int>& cumF,
                    int nFF, int sumT, FwdPairSet* out) {
    free_fwd_pairs(out);
    // LDS of a work-group: four share a compute unit.  Measured (lmax 10, 12 .. 3 channels,
    // B = 100: 24 KB 59 us, 32 KB 52 us, 40 KB 48 us, 53 KB 56 us).
    const size_t cap = 40 * 1024;
    // (l1, l2, n): a unit holds a degree once, the n-th repetition of a triple goes into a list of its own
    std::map<std::array<int, 3>, std::vector<PairTriple>> pairs;
    std::map<std::array<int, 3>, int> seen;
    for (const PairTriple& t : triples)
        if (t_F[t.l1] > 0 && t_F[t.l2] > 0) pairs[{t.l1, t.l2, seen[{t.l, t.l1, t.l2}]++}].push_back(t);
    struct Item { FwdPair u; size_t lds; double cost; };
    std::vector<Item> items;
    std::vector<FwdItem> its;
    for (auto& kv : pairs) {
        const int l1 = kv.first[0], l2 = kv.first[1];
        std::vector<PairTriple>& ts = kv.second;
        std::stable_sort(ts.begin(), ts.end(), [](const PairTriple& a, const PairTriple& b) { return a.l > b.l; });
        const int tau1 = t_F[l1], tau2 = t_F[l2];
        const int C = tau1 * tau2;
        std::vector<std::pair<int, int>> ranges;
        channel_ranges(C, tau2, &ranges);
        // Output degrees, largest first, in chunks of at most kPairNL whose work-group fits `cap` bytes (one degree always
        // goes): as few chunks as that allows, of about equal size.
        const int nt = (int)ts.size();
        FwdPair probe = FwdPair();
        probe.l1 = l1; probe.l2 = l2; probe.tau2 = tau2;
        set_channels(&probe, ranges[0]);
        const size_t front = pair_front_bytes(probe, probe.S);
        auto fits = [&](int b, int e) {
            size_t need = 0, most;
            for (int x = b; x < e; ++x) need += 512 * (size_t)(2 * ts[x].l + 1);
            return need + front + coef_bytes(l1, l2, ts[b].l, e - b, &most) <= cap;
        };
        std::vector<int> bounds;
        for (int nchunks = (nt + kPairNL - 1) / kPairNL;; ++nchunks) {
            bounds.assign(1, 0);
            for (int k = 0; k < nchunks && bounds.back() < nt; ++k) {
                const int b = bounds.back();
                int e = b + std::min(kPairNL, (nt - b + nchunks - k - 1) / (nchunks - k));
                while (e > b + 1 && !fits(b, e)) --e;
                bounds.push_back(e);
            }
            if (bounds.back() == nt) break;
        }
        for (size_t k = 0; k + 1 < bounds.size(); ++k) {
            const int b = bounds[k], e = bounds[k + 1];
            FwdPair first = FwdPair();                            // the items are the same for every channel range
            for (const auto& r : ranges) {
                Item it;
                FwdPair& u = it.u;
                u = FwdPair();
                u.l1 = l1; u.l2 = l2; u.nl = e - b;
                u.tau2 = tau2;
                set_channels(&u, r);
                u.offF1 = cumF[l1] + u.r0 * (2 * l1 + 1);
                u.offF2 = cumF[l2] + u.q0 * (2 * l2 + 1);
                size_t tile = 0;
                double terms = 0;
                for (int x = b; x < e; ++x) {
                    const PairTriple& t = ts[x];
                    const int M = 2 * t.l + 1;
                    u.l[x - b] = t.l;
                    u.cg[x - b] = t.cg;
                    u.offFF[x - b] = t.offFF + u.c0 * M;
                    u.chan[x - b] = t.chan0 + u.c0;
                    tile += 512 * (size_t)M;
                    terms += 2. * M * std::min(2 * l2 + 1, M);
                }
                for (int x = e - b; x < kPairNL; ++x) u.l[x] = -1;
                if (&r == &ranges[0]) {
                    make_items(&u, &its);
                    first = u;
                } else {
                    u.item0 = first.item0; u.cg_local = first.cg_local; u.cgbytes = first.cgbytes;
                    std::copy(first.wbeg, first.wbeg + kPairWaves + 1, u.wbeg);
                }
                it.lds = std::max(pair_front_bytes(u, u.S) + (size_t)u.cgbytes + tile, (size_t)u.nl * kPairWaves * 64 * 16);
                it.lds = align_up(it.lds, 16);
                it.cost = (terms + 4. * (2 * l1 + 1) * (2 * l2 + 1)) / u.S;
                if (it.lds > kPairMaxLds || pair_front_bytes(u, u.S) > 64 * 1024) return CGNET_OK;     // no units: never used
                items.push_back(it);
            }
        }
    }
    // one launch has one LDS size: units by the work-groups per compute unit their own need allows (five at most: beyond
    // that the registers decide), inside a class the dearest first
    auto cls = [](const Item& i) {
        return i.u.cg_local ? 0 : (int)std::max<size_t>(1, std::min<size_t>(4, kPairMaxLds / i.lds));
    };
    std::stable_sort(items.begin(), items.end(), [&](const Item& a, const Item& b) {
        return cls(a) != cls(b) ? cls(a) < cls(b) : a.cost > b.cost;
    });
    for (size_t k = 0; k < items.size(); ++k) {
        if (k == 0 || cls(items[k]) != cls(items[k - 1])) {
            out->class_begin.push_back((int)k);
            out->class_lds.push_back(0);
        }
        out->class_lds.back() = std::max(out->class_lds.back(), items[k].lds);
        out->lds = std::max(out->lds, items[k].lds);
        out->units.push_back(items[k].u);
        out->max_S = std::max(out->max_S, items[k].u.S);
    }
    out->class_begin.push_back((int)items.size());
    out->nFF = nFF;
    out->sumT = sumT;
    if (!out->units.empty()) {
        // units and items in one allocation, filled by one copy
        const size_t bytes = sizeof(FwdPair) * out->units.size(), at = align_up(bytes, 256), more = sizeof(FwdItem) * its.size();
        std::vector<unsigned char> tables(at + more);
        memcpy(tables.data(), out->units.data(), bytes);
        memcpy(tables.data() + at, its.data(), more);
        CGNET_HIP(hipMalloc((void**)&out->d_units, tables.size()));
        out->d_items = reinterpret_cast<FwdItem*>(reinterpret_cast<unsigned char*>(out->d_units) + at);
        CGNET_HIP(hipMemcpy(out->d_units, tables.data(), tables.size(), hipMemcpyHostToDevice));
        const void* kernels[] = {(const void*)cg_forward_pair_kernel<true, false>, (const void*)cg_forward_pair_kernel<false, false>,
                                 (const void*)cg_forward_pair_kernel<true, true>, (const void*)cg_forward_pair_kernel<false, true>};
        for (const void* k : kernels)
            if (int rc = raise_dynamic_lds(k, out->lds)) return rc;
    }
    return CGNET_OK;
}

void free_fwd_pairs(FwdPairSet* set) {
    if (set->d_units) (void)hipFree(set->d_units);
    *set = FwdPairSet();
}

int fwd_pairs_spg(const FwdPairSet& set, int B) {
    // Enough work-groups for a round and a half of the machine (four per compute unit), but as long as they last each
    // with samples for its lanes; eight stages at most, so that the last round is short.
    const int nu = std::max(1, (int)set.units.size());
    const int target = 1536;
    const int groups = std::max(1, std::min(B, (target + nu - 1) / nu));
    return std::min((B + groups - 1) / groups, std::max(8, set.max_S));
}

int launch_fwd_pairs(const FwdPairSet& set, const float* d_F, float* d_FF, const float* d_CG, int nF, int B, double* d_part,
                     int spg, hipStream_t s) {
    if (set.units.empty() || B == 0) return CGNET_OK;
    const int ngroups = (B + spg - 1) / spg;
    CGNET_REQUIRE((long long)set.units.size() * ngroups < (1LL << 31), CGNET_ERR_UNSUPPORTED,
                  "%zu units x %d sample groups exceed the grid limit", set.units.size(), ngroups);
    for (size_t k = 0; k + 1 < set.class_begin.size(); ++k) {
        const int u0 = set.class_begin[k], nu = set.class_begin[k + 1] - u0;
        const bool local = set.units[u0].cg_local != 0;
        auto launch = [&](auto* cg_forward_pair_kernel) {
            CGNET_LAUNCH(cg_forward_pair_kernel, dim3((unsigned)(nu * ngroups)), dim3(kPairThreads), set.class_lds[k], s,
                         (const float2*)d_F, (float2*)d_FF, d_CG, set.d_units + u0, set.d_items, nF, set.nFF, B, spg, d_part,
                         set.sumT);
        };
        if (d_part) launch(local ? &cg_forward_pair_kernel<true, true> : &cg_forward_pair_kernel<true, false>);
        else launch(local ? &cg_forward_pair_kernel<false, true> : &cg_forward_pair_kernel<false, false>);
        CGNET_HIP(hipGetLastError());
    }
    return CGNET_OK;
}

}  // namespace cgnet
