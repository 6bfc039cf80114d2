// Clebsch-Gordan product organised by pairs of input degrees (cg_pair.hip): types shared with the plans.
#pragma once
#include <vector>

#include "common.h"

namespace cgnet {

constexpr int kPairNL = 4;         // output degrees of one unit: the rows of a 4 x 4 x 1 matrix instruction
constexpr int kPairWaves = 4;      // waves of a work-group

// One work-group's share of a pair (l1, l2): up to kPairNL of its output degrees, a range of its channels.
// A lane of a wave is one channel (t1, t2) of one sample.
struct FwdPair {
    int l1, l2, nl;
    int c0, nc, S;                 // range of the pair's channels; samples a stage takes side by side (S * nc <= 64)
    int tau2;
    int r0, rows, q0, nt2;         // staged: rows [r0, r0 + rows) of degree l1, channels [q0, q0 + nt2) of degree l2
    int offF1, offF2;              // complex offsets of the staged rows inside a sample's F
    int cgbytes;                   // LDS bytes of the unit's coefficients
    int cg_local;                  // 0 = all items' coefficients at once, else bytes of one wave's buffer for one item
    int l[kPairNL];                // output degrees, largest first (-1: none)
    int cg[kPairNL];               // float offset of the triple's table
    int offFF[kPairNL];            // complex offset inside a sample's FF of channel c0
    int chan[kPairNL];             // channel c0 among all product channels (statistics)
    int item0;                     // the unit's items (FwdItem): wave w takes [item0 + wbeg[w], item0 + wbeg[w + 1])
    int wbeg[kPairWaves + 1];
    int pad[3];
};

// An item: the two values m, m + 1 of a unit's m axis.  Its steps are the m2 from lo on for which either has a term, in
// blocks of four and a last one of two (coefficients past the last term are zero).
struct FwdItem {
    int m8;                        // 8 m
    int fofs, gofs;                // byte offsets of F1[m - lo], F2[lo] from the entries of m1 = 0, m2 = 0
    int place;                     // byte offset of the item's coefficients
    int shape;                     // blocks of four | (1: two more steps) << 8 | degrees with both values << 16 |
                                   // (1: the next degree has m only, 2: m + 1 only) << 24
    int pad[3];
};

// Where a triple's channels lie in the product tensor the units write.
struct PairTriple { int l, l1, l2, cg, offFF, chan0; };

struct FwdPairSet {
    std::vector<FwdPair> units;
    FwdPair* d_units = nullptr;
    FwdItem* d_items = nullptr;
    std::vector<int> class_begin;      // units by the work-groups per compute unit their LDS allows: [begin[k], begin[k+1])
    std::vector<size_t> class_lds;
    size_t lds = 0;                    // largest class
    int max_S = 1;                     // most samples a unit takes side by side
    int nFF = 0, sumT = 0;             // complex entries / channels of one sample's product tensor
};

// `triples`: every kept triple with its place in the product tensor.  Leaves the set empty where a unit does not fit the LDS.
int build_fwd_pairs(const std::vector<PairTriple>& triples, const std::vector<int>& t_F, const std::vector<int>& cumF,
                    int nFF, int sumT, FwdPairSet* out);
void free_fwd_pairs(FwdPairSet* set);
int fwd_pairs_spg(const FwdPairSet& set, int B);       // samples per work-group
// d_part != nullptr: also the per-group partial statistics [group][sumT][2]
int launch_fwd_pairs(const FwdPairSet& set, const float* d_F, float* d_FF, const float* d_CG, int nF, int B, double* d_part,
                     int spg, hipStream_t s);

}  // namespace cgnet
