// cg_backward_pair_kernel: device code and launcher of one variant.  Every variant (KS groups of four output degrees, NT row tiles)
// is a translation unit of its own (cg_back_kernel_*.hip).
//
// With G_l = gFF of output degree l, the gradients of a pair (l1, l2) are
//     gF1[t1][m1] += sum_{t2, m2} H[t1, t2][m1, m2] conj F2[t2][m2],    gF2[t2][m2] += sum_{t1, m1} H[t1, t2][m1, m2] conj F1[t1][m1],
//     H[t1, t2][m1, m2] = sum_l C_l[m1 + m2][m2] G_l[t1, t2][m1 + m2].
// The fragments do not depend on l: all output degrees of a pair are gathered first (two real multiply-adds per entry, degree and
// value of m1 + m2), and the eight multiply-adds of the two gradients are spent once per (m1, m2) and not once per degree.
//
// A wave owns a unit: one pair, one sample, some of its channels (t1, t2).  It works on tiles of up to sixteen of them as columns and
// walks M = m1 + m2 upwards.  For one M, H is a product (m2 x l)(l x columns) on v_mfma_f32_16x16x4_f32: rows of the
// accumulator = sixteen values of m2 (up to three row tiles), steps of four degrees, left operand the packed coefficients as
// they lie in memory.  A lane then holds H for four m2 and one column and multiplies it on the vector ALUs: with F1[M - m2],
// summed over all M and tiles in registers (the gradient of degree l2), and with F2[m2], which belongs to m1 = M - m2.  Both
// the fragment F1[M - m2] and that second sum move by one row from one M to the next: four registers each in turn; a sum that
// has seen its four rows is added to LDS, where the other rows' shares of the same m1 and finally the columns of one t1 meet.
// Nothing is shared between waves and there is no barrier.
//
// G is taken in chunks of eight M in the layout of an accumulator (row = (M, re / im), column = channel), one register set per
// degree; four lane-group swaps per register set of four degrees turn it into right operands (lane group = degree).  It is read
// from memory (the stand-alone operator: sixteen segments of 64 bytes per load instruction) or, inside the layer, made from
// packed gO and packed weights by matrix instructions in the order of wmm_gradff_mfma_kernel, so that both sources hold the
// same values to the bit; where every degree has thirteen output channels or more, in bfloat16 pieces (split.h).
//
// Bounded by issue and latency: a vector multiply-add holds a SIMD for four cycles, an fp32 matrix instruction for 32, and the two take
// turns; a bfloat16 one for 16, four of them beside vector instructions.  lmax 11, 12 channels, B = 100, inside the layer: 8.6e7 vector
// and 1.13e7 fp32 matrix instructions, 75 % of the cycles of 1024 SIMDs at three waves a SIMD; lmax 20, 16 channels, in pieces: 59 % at two
// waves.  Three waves take 168 registers, and 41 more are spilled to 148 bytes of scratch a lane (41 .. 45 whatever the output channels, in
// pieces 36; up to lmax 7 128 registers, 5 or 6 spilled; none at lmax 12..15, 216 .. 254 registers, two waves; from lmax 16 on 256 registers,
// 26 .. 35 spilled): the kernel writes 161 MB there, of which 36 are partial gradients.  The loads of packed gO and weights come out of L1, which gives 64 bytes a
// cycle to loads of 4 or 16 bytes a lane and half of that to 8 bytes, and out of L2, for which the work-groups of a sample stay on one
// XCD.  Adding the sums in LDS with ds_add_f32 is no alternative to read and write: 18 times slower (measured alone).
// Against the kernels that work triple by triple, us (whole call, operands packed by itself): lmax 11, 12 channels, B = 100, layer
// 541 -> 416 (this kernel 391); lmax 20, 16 channels, B = 32, layer 4006 -> 2047 (G on fp32 instructions 2238); lmax 15, 16 channels, B = 64, stand-alone
// 1623 -> 1361; lmax 10, 4 channels, B = 100, stand-alone 106 -> 59.
#pragma once
#include <utility>

#include "cg_back_args.h"

namespace cgnet {
namespace {

typedef float v2f __attribute__((ext_vector_type(2)));
typedef float f32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));       // sixteen bytes on an 8-byte boundary
typedef __attribute__((address_space(3))) v2f* lds_v2_p;
typedef const __attribute__((address_space(3))) v2f* lds_cv2_p;

// the tables of a plan, read through the scalar cache
typedef const __attribute__((address_space(4))) BackPair* pair_p;
typedef const __attribute__((address_space(4))) BackGenPair* gen_pair_p;

__device__ __forceinline__ unsigned lds_address(const void* p) {
    return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
// complex entry k behind the LDS address a (a constant k becomes the instruction's offset)
__device__ __forceinline__ v2f lds_get(unsigned a, int k) { return ((lds_cv2_p)(uintptr_t)a)[k]; }
__device__ __forceinline__ void lds_put(unsigned a, int k, v2f v) { ((lds_v2_p)(uintptr_t)a)[k] = v; }
// f(0), f(1), ... f(N - 1) with constant arguments: arrays of registers are only ever indexed by constants
template <int N, typename F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>()), ...); }
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) { each_of<N>(f, std::make_integer_sequence<int, N>()); }
#define CGNET_EACH(N, I) each<N>([&](auto I##_) __attribute__((always_inline)) { constexpr int I = decltype(I##_)::value;
#define CGNET_END })

// LDS accesses of a wave are executed in order; this keeps the compiler from changing that order across lanes
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

// A copy the compiler knows nothing of: what is computed from it stays in the loop it is written in and takes no registers outside.
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// a pointer that is the same in all lanes, in scalar registers
__device__ __forceinline__ const float* uniform(const float* p) {
    const unsigned long long v = (unsigned long long)(uintptr_t)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (const float*)(uintptr_t)((unsigned long long)hi << 32 | lo);
}

// Four registers, lane groups of sixteen = four rows: register q, row a -> register a, row q.
__device__ __forceinline__ void swap32(float& x, float& y) {
    const auto z = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(z[0]);
    y = __uint_as_float(z[1]);
}
__device__ __forceinline__ void swap16(float& x, float& y) {
    const auto z = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(z[0]);
    y = __uint_as_float(z[1]);
}
__device__ __forceinline__ void turn_groups(f32x4 (&r)[4]) {
    CGNET_EACH(4, v)
        float r0 = r[0][v], r1 = r[1][v], r2 = r[2][v], r3 = r[3][v];
        swap32(r0, r2);
        swap32(r1, r3);
        swap16(r0, r1);
        swap16(r2, r3);
        r[0][v] = r0; r[1][v] = r1; r[2][v] = r2; r[3][v] = r3;
        __builtin_amdgcn_sched_barrier(0);
    CGNET_END;
}

// x / d for the small values here: inv = ceil(2^16 / d), d <= 16, x < 4096; inv = ceil(2^20 / d), d <= 47, x < 4096
__device__ __forceinline__ int div16(int x, int inv) { return (int)((unsigned)(x * inv) >> 16); }
__device__ __forceinline__ int div20(int x, int inv) { return (int)((unsigned)(x * inv) >> 20); }

// What a wave carries through its unit besides its accumulators.
struct BackWave {
    pair_p p;
    const float* w;                // layer source: the tile's packed weights, the sample's packed gO
    const float* go;
    const float* go_scales;
    const float2* gff;             // memory source: the sample's gFF
    const float* cp;               // coefficients of the current M
    int cstride;
    int w_group, go_chunk, go_degree;          // floats of a group of packed weights, of a chunk of packed gO, of a degree in it
    unsigned l8[kBackNL / 4];      // output degrees, a byte each: a table in memory would cost a wait before every fetch
    int lanes;                     // lanes that hold places of output channels
    int chan;                      // memory source: the lane's channel among those of the pair
    int last;                      // ... the last place in a sample with an entry behind it
    int lane, kk;
    unsigned f_at, s_at;           // LDS addresses: the lane's next row of F1, of the sums
};

// Two steps of four degrees: left operands (gO) and right operands (weights).  Loads of 4 or 16 bytes a lane run at 64 bytes a
// cycle out of L1, those of 8 bytes at half of that (measured): the weights come as two steps of two degrees a lane, gO step by step.
struct GenOps { float x[4][2]; f32x4 y[2]; };

// Where a group's operands lie: the weights in one run, the four degrees' gO.
struct GenAt { const f32x4* w; const float* go[4]; };

__device__ __forceinline__ GenAt gen_at(const BackWave& w, int group, const float* go_chunk) {
    GenAt at;
    at.w = reinterpret_cast<const f32x4*>(w.w + group * w.w_group);
    CGNET_EACH(4, q)
        at.go[q] = go_chunk + w.p->l[4 * group + q] * w.go_degree;
    CGNET_END;
    return at;
}

template <int S>
__device__ __forceinline__ void gen_load(const GenAt& at, int lane, GenOps& o) {
    CGNET_EACH(2, h) o.y[h] = (at.w + 64 * (2 * S + h))[lane]; CGNET_END;
    CGNET_EACH(4, q)
        o.x[q][0] = (at.go[q] + 128 * S)[lane];
        o.x[q][1] = (at.go[q] + 128 * S + 64)[lane];
    CGNET_END;
}

// n: the degrees of the group that reach the chunk; FIRST: sums begin
template <bool FIRST>
__device__ __forceinline__ void gen_steps(const GenOps& o, int n, f32x4 (&r)[4]) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    CGNET_EACH(4, q)
        if (q < n) {
            r[q] = mfma4(o.x[q][0], o.y[q / 2][2 * (q & 1)], FIRST ? zero : r[q]);
            r[q] = mfma4(o.x[q][1], o.y[q / 2][2 * (q & 1) + 1], r[q]);
        }
    CGNET_END;
}

// G of the chunk whose first value is M0 as right operands: r[group][M / 2][(M & 1, re / im)] in lane (degree of the group, column).
// Layer source with PAIRS pairs of steps over the output channels.  Places past the last degree that reaches the chunk keep what
// they held (their coefficients are zero).
template <int PAIRS, int KS>
__device__ __forceinline__ void back_make(const BackWave& w, int chunk, int nd, f32x4 (&r)[KS][4]) {
    {
        // a pair of steps is fetched while the one before it is multiplied
        const float* go = w.go + chunk * w.go_chunk;
        GenOps ops[2];
        GenAt at = gen_at(w, 0, go);
        gen_load<0>(at, w.lane, ops[0]);
        CGNET_EACH(KS, ks)
            const int n = nd - 4 * ks;                             // degrees of the group that reach the chunk
            if (n > 0) {
                const GenAt next = gen_at(w, n > 4 ? ks + 1 : ks, go);
                CGNET_EACH(PAIRS, s)
                    constexpr int now = (ks * PAIRS + s) & 1;
                    if constexpr (s + 1 < PAIRS) gen_load<s + 1>(at, w.lane, ops[1 - now]);
                    else gen_load<0>(next, w.lane, ops[1 - now]);
                    __builtin_amdgcn_sched_barrier(0);
                    gen_steps<s == 0>(ops[now], n, r[ks]);
                CGNET_END;
                at = next;
            }
        CGNET_END;
    }
}

// The same from operands in pieces.
struct SplitOps { bf16x8 a[kPieces], b[kPieces]; };

template <int KS>
__device__ __forceinline__ void back_make_split(const BackWave& w, int chunk, int nd, f32x4 (&r)[KS][4]) {
    // The operands of a degree are fetched while those of the one before it are multiplied (places past the last degree: whatever
    // lies there).
    SplitOps ops[2] = {};
    const bool on = w.lane < w.lanes;                              // places past the output channels stay zero
    const float *go = w.go + kBackOperand * chunk, *wt = uniform(w.w);
    const v2f scale = *reinterpret_cast<const v2f*>(w.go_scales + kBackScales * chunk + 2 * w.kk);
    auto load = [&](auto k, SplitOps& o) __attribute__((always_inline)) {
        const unsigned l = (w.l8[k / 4] >> (8 * (k % 4))) & 255u;
        if (on) {
            CGNET_EACH(kPieces, i) o.b[i] = reinterpret_cast<const bf16x8*>(wt + kBackOperand * k)[64 * i + w.lane]; CGNET_END;
            CGNET_EACH(kPieces, i) o.a[i] = reinterpret_cast<const bf16x8*>(go + l * (unsigned)w.go_degree)[64 * i + w.lane]; CGNET_END;
        }
    };
    load(std::integral_constant<int, 0>(), ops[0]);
    CGNET_EACH(4 * KS, q)
        if (q < nd) {
            if constexpr (q + 1 < 4 * KS) load(std::integral_constant<int, q + 1>(), ops[1 - (q & 1)]);
            __builtin_amdgcn_sched_barrier(0);
            const SplitOps& o = ops[q & 1];
            const f32x4 z = split_product(o.a, o.b);
            r[q / 4][q % 4] = (f32x4){z[0] * scale.x, z[1] * scale.x, z[2] * scale.y, z[3] * scale.y};
        }
    CGNET_END;
}

// Memory source: entries M0 + 2 kk, M0 + 2 kk + 1 of the lane's channel, degree k of the pair.  Where one of them is no value of the
// degree its place may hold any entry of the sample: its coefficients are zero.  So are those of a place past the last degree
// that reaches the chunk, which repeats it.
__device__ __forceinline__ int mem_at(const BackWave& w, int M0, int k, int nd) {
    const int q = min(k, nd - 1), l = w.p->l[q];
    const int i = max(-1, min(M0 + 2 * w.kk + l, 2 * l));
    return __mul24(w.chan, 2 * l + 1) + (i + w.p->offFF[q]);
}
__device__ __forceinline__ f32x4 mem_load(const BackWave& w, int M0, int k, int nd) {
    const int at = max(0, min(mem_at(w, M0, k, nd), w.last));     // the first and the last entry of a sample have one neighbour
    return *reinterpret_cast<const f32x4_a8*>(reinterpret_cast<const char*>(w.gff) + 8u * (unsigned)at);
}
// after the loads of a chunk of a tile that holds the first or the last channel of a sample
template <int KS>
__device__ __forceinline__ void mem_ends(const BackWave& w, int M0, int nd, f32x4 (&r)[KS][4]) {
    CGNET_EACH(4 * KS, k)
        const int at = mem_at(w, M0, k, nd);
        const f32x4 z = r[k / 4][k % 4];
        r[k / 4][k % 4] = (f32x4){at > w.last ? z[2] : z[0], at > w.last ? z[3] : z[1], at < 0 ? z[0] : z[2], at < 0 ? z[1] : z[3]};
    CGNET_END;
}

template <int KS>
__device__ __forceinline__ void turn_all(int nd, f32x4 (&r)[KS][4]) {
    CGNET_EACH(KS, ks)
        if (4 * ks < nd) turn_groups(r[ks]);
        __builtin_amdgcn_sched_barrier(0);
    CGNET_END;
}

// Accumulators of a wave: f2, a2: entries and gradients of degree l2 (row tile, row); f1, s1: slot M & 3 holds F1[M - m2] and the
// sum of m1 = M - m2, m2 the lane's first row of the tile.
template <int NT>
struct BackAcc {
    float f2r[NT][4], f2i[NT][4], a2r[NT][4], a2i[NT][4], s1r[NT][4], s1i[NT][4];
    v2f f1[NT][4];
};

// A chunk of eight M with at most KC groups of degrees.  AHEAD (memory source): the loads of the chunk at next_M0 with next_nd degrees
// go out between the steps, behind the coefficients of the step after, so that no wait for those is one for all of them.
template <int KS, int NT, int KC, bool AHEAD>
__device__ __forceinline__ void back_chunk(BackWave& w, BackAcc<NT>& A, const f32x4 (&G)[KS][4], int steps8, int tiles8,
                                           f32x4 (&next)[KS][4], int next_M0, int next_nd) {
    float cf[2][KC][NT];
    CGNET_EACH(KC, ks) CGNET_EACH(NT, rt) cf[0][ks][rt] = (w.cp + (ks * NT + rt) * 64)[w.lane]; CGNET_END; CGNET_END;
    lds_order();                                                   // keeps the loads here and not where they are used
    CGNET_EACH(8, x)
        const int nk = (steps8 >> (4 * x)) & 15, tm = (tiles8 >> (4 * x)) & 15;
        constexpr int now = x & 1, slot = x & 3, done = (x + 1) & 3;
        v2f old[NT];
        CGNET_EACH(NT, rt)
            A.f1[rt][slot] = lds_get(w.f_at, x + 16 * (NT - 1 - rt) + 3);
            old[rt] = lds_get(w.s_at, kBackPitch * (x + 16 * (NT - 1 - rt)));
        CGNET_END;
        w.cp += w.cstride;
        if constexpr (x < 7) {
            CGNET_EACH(KC, ks) CGNET_EACH(NT, rt) cf[1 - now][ks][rt] = (w.cp + (ks * NT + rt) * 64)[w.lane]; CGNET_END; CGNET_END;
        }
        if constexpr (AHEAD) {
            constexpr int per = KS / 2 + (KS & 1);                 // 4 KS loads in eight steps
            CGNET_EACH(per, y)
                if constexpr (per * x + y < 4 * KS)
                    next[(per * x + y) / 4][(per * x + y) % 4] = mem_load(w, next_M0, per * x + y, next_nd);
            CGNET_END;
        }
        CGNET_EACH(NT, rt)
            if (tm & (1 << rt)) {
                const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
                f32x4 hr = mfma4(cf[now][0][rt], G[0][x / 2][2 * now], zero);
                f32x4 hi = mfma4(cf[now][0][rt], G[0][x / 2][2 * now + 1], zero);
                CGNET_EACH(KC - 1, k)
                    if (k + 1 < nk) {
                        hr = mfma4(cf[now][k + 1][rt], G[k + 1][x / 2][2 * now], hr);
                        hi = mfma4(cf[now][k + 1][rt], G[k + 1][x / 2][2 * now + 1], hi);
                    }
                CGNET_END;
                CGNET_EACH(4, v)
                    constexpr int s = (x - v) & 3;
                    A.a2r[rt][v] = fmaf(hr[v], A.f1[rt][s].x, A.a2r[rt][v]);
                    A.a2i[rt][v] = fmaf(hi[v], A.f1[rt][s].x, A.a2i[rt][v]);
                    A.s1r[rt][s] = v == 0 ? hr[v] * A.f2r[rt][v] : fmaf(hr[v], A.f2r[rt][v], A.s1r[rt][s]);
                    A.s1i[rt][s] = v == 0 ? hi[v] * A.f2r[rt][v] : fmaf(hi[v], A.f2r[rt][v], A.s1i[rt][s]);
                    A.a2r[rt][v] = fmaf(hi[v], A.f1[rt][s].y, A.a2r[rt][v]);
                    A.a2i[rt][v] = fmaf(-hr[v], A.f1[rt][s].y, A.a2i[rt][v]);
                    A.s1r[rt][s] = fmaf(hi[v], A.f2i[rt][v], A.s1r[rt][s]);
                    A.s1i[rt][s] = fmaf(-hr[v], A.f2i[rt][v], A.s1i[rt][s]);
                CGNET_END;
            } else {
                A.s1r[rt][slot] = A.s1i[rt][slot] = 0.f;
            }
            lds_put(w.s_at, kBackPitch * (x + 16 * (NT - 1 - rt)), (v2f){old[rt].x + A.s1r[rt][done], old[rt].y + A.s1i[rt][done]});
        CGNET_END;
        lds_order();
    CGNET_END;
    w.f_at += 64u;
    w.s_at += 64u * kBackPitch;
}

template <int KS, int NT, int SOURCE>
__device__ __forceinline__ void back_unit(const BackArgs& a, pair_p p, const BackUnit& u, int b, float* lds, int lane) {
    const int j = lane & 15, kk = lane >> 4;
    const int l1 = p->l1, l2 = p->l2, M1 = 2 * l1 + 1, M2 = 2 * l2 + 1, tau2 = p->tau2, nrows = p->nrows;
    const int rows = back_rows(p->nch, NT), pitch = back_row_pitch(rows);
    const int M0 = a.grid0 + 8 * p->c0;
    const int row0 = -l1 - (M0 + l2 - 16 * NT + 1);                // row of m1 = -l1
    v2f* const sums = reinterpret_cast<v2f*>(lds);
    v2f* const zeros = sums + rows * kBackPitch - kBackSpare;
    v2f* const f1buf = zeros + pitch - 1;                          // [nbuf][nrows][pitch]
    const int C = p->tau1 * tau2;
    const int inv2 = p->inv_tau2;
    const int first2 = u.tile0 * p->ncol - div16(u.tile0 * p->ncol, inv2) * tau2;     // t2 of the first column
    const int t2 = first2 + j - div16(first2 + j, inv2) * tau2;
    {
        f32x4* z = reinterpret_cast<f32x4*>(lds);
        const int n = back_lds_floats(p->nch, NT, nrows, p->nbuf) >> 2;
        for (int e = lane; e < n; e += 64) z[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // the zeros precede the copies
    const float2* Fb = a.F + (size_t)b * a.nF;
    auto stage = [&](int tile, int buf) {                          // the tile's rows of degree l1
        const int ln = opaque(lane);
        const int r = div16(tile * p->ncol, inv2), n = min(nrows, p->tau1 - r);
        const float* src = reinterpret_cast<const float*>(Fb + p->offF1 + r * M1);
        for (int k = 0; k < n; ++k) {
            float* dst = reinterpret_cast<float*>(f1buf + (buf * nrows + k) * pitch + row0);
            for (int x = 0; x < 2 * M1; x += 64)
                if (x + ln < 2 * M1)
                    __builtin_amdgcn_global_load_lds(src + k * 2 * M1 + x + ln, (lds_void_ptr)(dst + x), 4, 0, 0);
        }
    };
    stage(u.tile0, 0);
    BackAcc<NT> A;
    CGNET_EACH(NT, rt) CGNET_EACH(4, v)
        const int m = 16 * rt + 4 * kk + v;
        float2 z = make_float2(0.f, 0.f);
        if (j < p->ncol && m < M2) z = Fb[p->offF2 + t2 * M2 + m];
        A.f2r[rt][v] = z.x;
        A.f2i[rt][v] = z.y;
        A.a2r[rt][v] = A.a2i[rt][v] = 0.f;
    CGNET_END; CGNET_END;
    f32x4 G[KS][4];
    CGNET_EACH(KS, ks) CGNET_EACH(4, q) G[ks][q] = (f32x4){0.f, 0.f, 0.f, 0.f}; CGNET_END; CGNET_END;
    BackWave w;
    w.p = p;
    const gen_pair_p g = (gen_pair_p)(uintptr_t)(SOURCE != kBackMemory ? a.gp + u.pair : nullptr);
    w.w_group = 512 * SOURCE;
    w.go_scales = SOURCE == kBackSplit ? a.Go + (size_t)b * a.nGo + a.go_scales : nullptr;
    w.lanes = a.lanes;
    CGNET_EACH(kBackNL / 4, q) w.l8[q] = p->l8[q]; CGNET_END;
    w.go_chunk = a.go_chunk;
    w.go_degree = a.go_degree;
    w.go = SOURCE != kBackMemory ? a.Go + (size_t)b * a.nGo : nullptr;
    w.gff = SOURCE != kBackMemory ? nullptr : a.gFF + (size_t)b * a.nFF;
    w.cstride = p->nks * NT * 64;
    w.last = a.nFF - 2;
    w.lane = lane;
    w.kk = kk;
    const unsigned lane_row = 8u * (unsigned)(4 * (3 - kk));       // the lane's first row, in complex entries of one column
    const unsigned s_base = lds_address(sums) + kBackPitch * lane_row + 8u * (unsigned)j;

    for (int k = 0; k < u.ntiles; ++k) {
        const int tile = u.tile0 + k * p->tstep, buf = k & 1;
        const int c0 = tile * p->ncol, first = div16(c0, inv2);    // the tile's first channel and row
        const int ncol = min(p->ncol, C - c0), nr = div16(c0 + ncol - 1, inv2) - first + 1;
        const int jj = opaque(j), t1 = div16(c0 + jj, inv2);       // lanes past the last column: a row of zeros
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // the tile's rows of degree l1 have landed
        if (k + 1 < u.ntiles) stage(tile + p->tstep, buf ^ 1);
        w.f_at = lds_address(jj < ncol ? f1buf + (buf * nrows + t1 - first) * pitch : zeros) + lane_row;
        w.s_at = s_base;
        CGNET_EACH(NT, rt) CGNET_EACH(3, v)
            A.f1[rt][3 - v] = lds_get(w.f_at, 16 * (NT - 1 - rt) + 2 - v);
            A.s1r[rt][3 - v] = A.s1i[rt][3 - v] = 0.f;
        CGNET_END; CGNET_END;
        w.w = SOURCE != kBackMemory ? a.W + (g->w + tile * g->wtile) : nullptr;
        // memory source: a lane past the last channel repeats the last row's of its t2
        if constexpr (SOURCE == kBackMemory) w.chan = min(t1, p->tau1 - 1) * tau2 + (t1 < p->tau1 ? c0 + jj - t1 * tau2 : t2);
        // all loads of a chunk go out during the one before it where there are registers for them
        constexpr bool AHEAD = SOURCE == kBackMemory && KS + NT <= 6;
        const bool ends = (p->ends & 1 && c0 == 0) || (p->ends & 2 && c0 + ncol == C);
        f32x4 next[KS][4];
        if constexpr (AHEAD) {
            CGNET_EACH(4 * KS, q) next[q / 4][q % 4] = mem_load(w, M0, q, p->degs[0]); CGNET_END;
        }
        w.cp = a.coef + p->coef;
        for (int c = 0; c < p->nch; ++c) {
            const int steps8 = p->steps[c], tiles8 = p->tiles[c], nd = p->degs[c];
            const int Mc = M0 + 8 * c, c1 = min(c + 1, p->nch - 1), next_M0 = M0 + 8 * c1, next_nd = p->degs[c1];
            if constexpr (SOURCE == kBackSplit) {
                back_make_split<KS>(w, p->c0 + c, nd, G);
            } else if constexpr (SOURCE > 0) {
                back_make<SOURCE, KS>(w, p->c0 + c, nd, G);
            } else {
                CGNET_EACH(4 * KS, q)
                    if constexpr (AHEAD) G[q / 4][q % 4] = next[q / 4][q % 4];
                    else if (q < nd + 3) G[q / 4][q % 4] = mem_load(w, Mc, q, nd);
                CGNET_END;
                if (ends) mem_ends<KS>(w, Mc, nd, G);
            }
            turn_all<KS>(nd, G);
            if (nd <= 4) back_chunk<KS, NT, 1, AHEAD>(w, A, G, steps8, tiles8, next, next_M0, next_nd);
            else if (KS == 2 || nd <= 8) back_chunk<KS, NT, 2, AHEAD>(w, A, G, steps8, tiles8, next, next_M0, next_nd);
            else back_chunk<KS, NT, KS, AHEAD>(w, A, G, steps8, tiles8, next, next_M0, next_nd);
        }
        // the three sums that have not seen their last row
        CGNET_EACH(3, x)
            CGNET_EACH(NT, rt)
                const int at = kBackPitch * (x + 16 * (NT - 1 - rt));
                const v2f o = lds_get(w.s_at, at);
                lds_put(w.s_at, at, (v2f){o.x + A.s1r[rt][(x + 1) & 3], o.y + A.s1i[rt][(x + 1) & 3]});
            CGNET_END;
            lds_order();
        CGNET_END;
        // gradient of the tile's rows of degree l1: the columns of a row t1 added in order
        const int ln = opaque(lane);
        float2* p1 = a.part + (size_t)b * a.P + u.p1off + k * nrows * M1;
        for (int e = ln; e < nr * M1; e += 64) {
            const int r = div20(e, p->inv_M1), x = e - r * M1;
            const int from = max(0, (first + r) * tau2 - c0), to = min(ncol, (first + r + 1) * tau2 - c0);
            const v2f* col = sums + (row0 + x) * kBackPitch;
            float2 s = make_float2(0.f, 0.f);
            for (int t = from; t < to; ++t) {
                s.x += col[t].x;
                s.y += col[t].y;
            }
            p1[e] = s;
        }
        lds_order();
        {
            // (the rows of no m1 hold sums of zeros)
            f32x4* z = reinterpret_cast<f32x4*>(sums + row0 * kBackPitch);
            for (int e = ln; e < M1 * (kBackPitch / 2); e += 64) z[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
        lds_order();
    }
    // gradient of degree l2: the tiles are in the registers, columns of one t2 lie tau2 apart
    CGNET_EACH(NT, rt) CGNET_EACH(4, v)
        sums[(16 * rt + 4 * kk + v) * kBackPitch + j] = (v2f){A.a2r[rt][v], A.a2i[rt][v]};
    CGNET_END; CGNET_END;
    lds_order();
    float2* p2 = a.part + (size_t)b * a.P + u.p2off;
    const int repeats = div16(p->ncol + tau2 - 1, inv2);
    for (int e = opaque(lane); e < tau2 * M2; e += 64) {
        const int t = div20(e, p->inv_M2), m = e - t * M2;
        const int c = t - first2 + (t < first2 ? tau2 : 0);
        const v2f* from = sums + m * kBackPitch + c;
        float2 s = make_float2(0.f, 0.f);
        for (int r = 0; r < repeats; ++r)
            if (c + r * tau2 < p->ncol) {
                s.x += from[r * tau2].x;
                s.y += from[r * tau2].y;
            }
        p2[e] = s;
    }
}

template <int KS, int NTMAX, int SOURCE>
__global__ void __launch_bounds__(kBackThreads, SOURCE == kBackMemory ? (NTMAX == 1 ? 3 : 2) : NTMAX == 1 ? 4 : KS + NTMAX <= 5 ? 3 : 2)
cg_backward_pair_kernel(BackArgs a) {
    extern __shared__ __align__(16) float back_lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    // Work-groups go round the eight XCDs in turn.  All units of four samples run on the same one, whose L2 then holds the packed gO
    // of an eighth of the batch; the samples left over come first and go everywhere.
    const int quads = (a.B + kBackWaves - 1) / kBackWaves, left = quads & 7, spread = a.nunits * left;
    const bool pinned = (int)blockIdx.x >= spread;
    const int at = pinned ? (int)blockIdx.x - spread : (int)blockIdx.x, per_unit = pinned ? quads - left : left;
    const int unit = at / per_unit, b = (at - unit * per_unit + (pinned ? left : 0)) * kBackWaves + wave;
    if (b >= a.B) return;
    const auto* up4 = (const __attribute__((address_space(4))) int*)(uintptr_t)(a.units + unit);
    const BackUnit u = {up4[0], up4[1], up4[2], up4[3], up4[4]};
    const pair_p p = (pair_p)(uintptr_t)(a.pairs + u.pair);
    float* lds = back_lds + wave * a.lds_wave;
    if (NTMAX == 1 || p->nt == 1) back_unit<KS, 1, SOURCE>(a, p, u, b, lds, lane);
    else if (NTMAX == 2 || p->nt == 2) back_unit<KS, NTMAX >= 2 ? 2 : 1, SOURCE>(a, p, u, b, lds, lane);
    else back_unit<KS, NTMAX, SOURCE>(a, p, u, b, lds, lane);
}

template <int KS, int NT>
const void* back_kernel(int source) {
    return source == 0   ? (const void*)cg_backward_pair_kernel<KS, NT, 0>
           : source == 1 ? (const void*)cg_backward_pair_kernel<KS, NT, 1>
           : source == 2 ? (const void*)cg_backward_pair_kernel<KS, NT, 2>
           : source == 3 ? (const void*)cg_backward_pair_kernel<KS, NT, 3>
           : source == 4 ? (const void*)cg_backward_pair_kernel<KS, NT, 4>
                         : (const void*)cg_backward_pair_kernel<KS, NT, kBackSplit>;
}

template <int KS, int NT>
void back_launch(int source, dim3 grid, size_t lds, hipStream_t s, const BackArgs& a) {
    auto launch = [&](auto* cg_backward_pair_kernel) {
        CGNET_LAUNCH(cg_backward_pair_kernel, grid, dim3(kBackThreads), lds, s, a);
    };
    switch (source) {
        case 0: launch(&cg_backward_pair_kernel<KS, NT, 0>); break;
        case 1: launch(&cg_backward_pair_kernel<KS, NT, 1>); break;
        case 2: launch(&cg_backward_pair_kernel<KS, NT, 2>); break;
        case 3: launch(&cg_backward_pair_kernel<KS, NT, 3>); break;
        case 4: launch(&cg_backward_pair_kernel<KS, NT, 4>); break;
        default: launch(&cg_backward_pair_kernel<KS, NT, kBackSplit>); break;
    }
}

}  // namespace

#define CGNET_BACK_VARIANT(V, KS, NT)                                                                              \
    const void* back_kernel_##V(int source) { return back_kernel<KS, NT>(source); }                                  \
    void back_launch_##V(int source, dim3 grid, size_t lds, hipStream_t s, const BackArgs& a) {                     \
        back_launch<KS, NT>(source, grid, lds, s, a);                                                               \
    }

}  // namespace cgnet
