// Host-side functions the translation units of libcgnet_hip call in each other (not part of the C ABI).
#pragma once
#include <algorithm>

#include "common.h"
#include "cg_plan.h"
#include "wmm_plan.h"

namespace cgnet {

// ---- fnwmm.hip
size_t wmm_forward_wp_bytes(const cgnet_wmm_plan* plan);              // packed forward weights
size_t wmm_forward_opart_bytes(const cgnet_wmm_plan* plan, int B);    // partial outputs of the channel slices
// O = W' FF with the weights already packed (pack_w_forward_thread); d_opart: wmm_forward_opart_bytes bytes
int wmm_forward_packed(const cgnet_wmm_plan* plan, const float* d_FF, float* d_O, const float* d_Wp, int B,
                       void* d_opart, hipStream_t s);

// raw weight-gradient sums  sum_{b in chunk, m} gO conj(FF)  per chunk of samples: d_part[chunk][nW] complex
// (wmm_gradw_part_bytes bytes); *nchunks = chunks written.  The caller adds them and divides by the stds.
size_t wmm_gradw_part_bytes(const cgnet_wmm_plan* plan, int B);
int wmm_gradw_raw(const cgnet_wmm_plan* plan, const float* d_gO, const float* d_FF, float* d_part, int B, int* nchunks,
                  hipStream_t s);

// ---- cg_product.hip
int cg_forward_spg(const cgnet_cg_plan* p, int B);       // samples per work-group of the product forward
// the product kernels of one call; d_part != nullptr: also the per-group partial statistics [group][sumT][2]
// d_tasks: another table of the plan's forward tasks, in the same order, whose tiles lie elsewhere in the product
// tensor (nFF complex entries and sumT channels per sample); nullptr = the plan's own
int cg_launch_forward(const cgnet_cg_plan* p, const float* d_F, float* d_FF, const float* d_CG, int B, double* d_part,
                      int spg, hipStream_t s, const CgTask* d_tasks = nullptr, int nFF = 0, int sumT = 0);
// Per-task metadata of the fused layer backward for this pair of plans, on the current device.  link->ok says
// whether the fused kernel takes the pair; when it does not, the return code is CGNET_ERR_UNSUPPORTED and
// cgnet_last_error() names the reason.
int build_fused_link(const cgnet_cg_plan* p, const cgnet_wmm_plan* w, FusedLink* link);
void free_fused_link(FusedLink* link);
// bytes of the unit backward's own areas (partials, padded fragments, padded tables) = cgnet_sparse_backward_workspace
struct BwdAreas { size_t part1, part2, Fp, CGP, total; };
BwdAreas bwd_areas(const cgnet_cg_plan* p, int B);
// padded fragments and tables (the operands the unit kernels copy into LDS)
int launch_backward_pad(const cgnet_cg_plan* p, const float* d_F, const float* d_CG, float* d_Fp, float* d_CGP, int B,
                        hipStream_t s);
// packed A operand (conj-free weights / div, per task) of the fused backward
int launch_pack_w_gen(const FusedLink& link, const float* d_W, const float* d_stds, float eps, float* d_Ag, hipStream_t s);
// gO packing + fused kernel + combine; the A operand, padded fragments and tables are given
int launch_fused_backward(const cgnet_cg_plan* p, const FusedLink& link, const float* d_gO, const float* d_Ag,
                          const float* d_Fp, const float* d_CGP, float* d_Bg, float* d_part1, float* d_part2,
                          float* d_gF, int B, hipStream_t s);

int launch_zero_gradient(const cgnet_cg_plan* p, float* d_gF, int B, hipStream_t s);      // a fill kernel: may be recorded

// ---- cg_back.hip: backward by pairs of input degrees
// `triples`: every kept triple with its place in the product tensor.  Leaves the set empty where the shape is not taken.
int build_back_set(const std::vector<PairTriple>& triples, const std::vector<int>& t_F, const std::vector<int>& cumF, int L, int nFF,
                   BackSet* out);
void free_back_set(BackSet* set);
const BackLevel& back_level(const BackSet& set, int B);              // the cut for a batch of B samples
// Bytes that serve a batch of B samples and every smaller one, from bytes(b), those of b samples alone.  A smaller batch may take a
// finer cut (more partial gradients a sample) or, up to most_B samples, go by pairs where this one does not: in between bytes(b)
// grows with b.
template <typename Bytes>
size_t back_bytes_up_to(const BackSet& set, int most_B, int B, Bytes&& bytes) {
    size_t most = bytes(B);
    auto look = [&](int b) { if (b >= 1 && b < B) most = std::max(most, (size_t)bytes(b)); };
    if (!set.ok()) return most;
    look(most_B);
    for (const BackLevel& lv : set.levels)
        if (lv.least_B - 1 <= most_B) look(lv.least_B - 1);
    return most;
}
// Largest batch the backward by pairs is taken for, against a kernel that works triple by triple.  By pairs a call ends earlier
// however few samples it has; where a pair has few output degrees, or rows and columns of its tiles are empty, the other spends
// less on a sample, and large batches show it.  Both sides are sums over a sample's work, the constants fitted to the choice
// (not to the times: a rule's terms are right up to a common factor) over lmax 3..23, 1..16 channels (constant and falling with
// the degree), default and minimum-spanning-tree (MST) triples, 1..128 samples, 5447 calls of 25 us and more:
//   stand-alone, hybrid kernel   by the rule 0.67 of the time triple by triple, 0.3 % of the calls more than 5 % slower, at worst
//                                1.12 times; always by pairs 0.75, 33 %, 2.55 times
//   stand-alone, unit kernel     by the rule 0.59, 0.6 %, 1.16 times; always 0.60, 8 %, 1.66 times
//   layer, 8..16 channels        by the rule 0.62, 1.4 %, 1.26 times (lmax 16, MST, 11 channels, B = 128: 1090 -> 1376 us); always
//                                0.63, 14 %, 1.64 times
//     (G on fp32 instructions; in pieces (split.h), over 36 layers of MST triples, lmax 8..20, 9..15 channels
//     in and out, 8..128 samples: triples are the faster wherever the rule takes them, pairs at worst 1.12 times, lmax 11, 9 channels, B = 32)
// A layer with other channels has no other kernel but the two of the chain: always by pairs, 0.48 of their time, 0.3 % of 2325 calls
// slower, at worst 1.14 times.
struct BackRule {
    double block, tile;            // 1e-4 us of a sample by pairs: per block of 16 x 16 entries of H, per tile of channels
    double mac, entry, task;       // ... triple by triple: per multiply-add, per entry of the product, per task of a unit
    double start, start_L2;        // us that a small batch saves: at lmax 0, times lmax squared
};
constexpr BackRule kBackRuleUnit = {3.0, 49., 0.0095, 0., 15.7, 16., 0.186};
constexpr BackRule kBackRuleHybrid = {1.8, 37., 0., 0.041, 13., 8., 0.21};
constexpr BackRule kBackRuleLayer = {1.2, 46., 0., 0.059, 51., 13., 0.04};
int back_most_batch(const BackSet& set, int L, int nFF, int ntasks, const BackRule& rule);
int launch_pack_coef_back(const BackSet& set, const float* d_CG, float* d_coef, hipStream_t s);
// d_part: lv.P * B complex entries for the partial gradients, which are added up to d_gF
int launch_back_memory(const BackSet& set, const BackLevel& lv, const float* d_F, const float* d_gFF, const float* d_coef,
                       float* d_part, float* d_gF, int L, int nF, int nFF, int B, hipStream_t s);
// The same with the gradient of the product made in registers from packed weights and gO.  link->ok says whether the pair of
// plans is taken; when it is not, the return code is CGNET_ERR_UNSUPPORTED and cgnet_last_error() names the reason.
int build_back_link(const cgnet_cg_plan* p, const cgnet_wmm_plan* w, BackLink* link);
void free_back_link(BackLink* link);
int launch_pack_w_back(const BackLink& link, const float* d_W, const float* d_stds, float eps, float* d_Wp, hipStream_t s);
int launch_back_layer(const BackSet& set, const BackLink& link, const BackLevel& lv, const float* d_F, const float* d_gO,
                      const float* d_Wp, const float* d_coef, float* d_Go, float* d_part, float* d_gF, int L, int nF, int B,
                      hipStream_t s);

// ---- fused inference forward (cg_product.hip)
int build_fwd_link(const cgnet_cg_plan* p, const cgnet_wmm_plan* w, FwdLink* link);
void free_fwd_link(FwdLink* link);
int launch_pack_w_mix(const cgnet_cg_plan* p, const FwdLink& link, const float* d_W, const float* d_stds, float eps, float* d_Af,
                      hipStream_t s);
// product tiles mixed in LDS + the sum of the tasks' partial outputs; d_Opart: link.opart * B complex entries
int launch_forward_fused(const cgnet_cg_plan* p, const FwdLink& link, const float* d_F, const float* d_CG, const float* d_Af,
                         float* d_Opart, float* d_O, int B, hipStream_t s);

}  // namespace cgnet
