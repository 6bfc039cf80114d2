"""The product forward organised by pairs of input degrees (cg_forward_pair_kernel) where its pieces have edges: channel
ranges of a lane-width and one over, lanes shared by several samples with a short last stage, one output degree per unit,
rows beyond one copy instruction, coefficients that do not fit the LDS, a triple kept twice, empty degrees.  Same tolerance
as tests/test_gpu_parity.py: the strict bar, or three times what float32 arithmetic on the CPU is off by."""
import pytest
import torch

from tests.test_gpu_parity import F32, assert_close, cg_oracle_fwd_bwd, dev, edge_pairs, make_codes, rand_straight  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    # lmax, taus, B, triples
    (0, [3], 5, "default"),
    (2, [1, 1, 1], 67, "default"),                                    # 64 samples in a stage, then three
    (4, [5, 13, 5, 1, 16], 4, "default"),                             # 65 channels, 64 + 1 and 16 x 16 among the ranges
    (6, [4, 0, 16, 4, 1, 3, 7], 9, "default"),                        # an empty degree, ranges of whole waves
    (9, [12, 7, 6, 5, 4, 4, 4, 3, 3, 3], 7, "mst"),
    (15, [2] * 16, 6, "mst"),
    (18, [1, 3] * 9 + [1], 4, "mst"),                                 # rows longer than one copy instruction
    (26, [2, 1] * 13 + [2], 4, "edge"),                               # coefficients fetched item by item
    (3, [2, 3, 1, 2], 11, [[(1, 1)], [(1, 1), (2, 1), (2, 1)], [(2, 2), (2, 2), (3, 1)], [(3, 0)]]),   # kept twice
]


@pytest.mark.parametrize("lmax,taus,bsz,mode", CASES)
def test_pair_forward_and_statistics(dev, lmax, taus, bsz, mode):  # noqa: F811
    from cgnet_amd import CG_layers, _lib
    pairs = edge_pairs(lmax) if mode == "edge" else mode
    mod = CG_layers.CG_woFilter_cuda(lmax, taus, lll_mode=None if mode == "default" else pairs, device=dev)
    codes = mod.lll_list
    plan = mod.native_plan()
    x64 = rand_straight(taus, bsz, seed=lmax + bsz)
    want, _ = cg_oracle_fwd_bwd(lmax, taus, codes, x64)
    twin, _ = cg_oracle_fwd_bwd(lmax, taus, codes, x64, dtype=F32)
    x = x64.float().to(dev)
    lib = _lib.load()
    lib.cgnet_profile_reset()
    lib.cgnet_profile_enable(1)
    y = mod(x, straight_output=True)
    torch.cuda.synchronize()
    lib.cgnet_profile_enable(0)
    assert set(_lib.kernel_times()) == {"cg_forward_pair_kernel"}
    assert_close(y, want, "pair forward", twin)
    ff = torch.full_like(y, float("nan"))
    sums = torch.full((plan.sum_tFF, 2), float("nan"), device=dev, dtype=torch.float64)
    plan.forward_stats(x, ff, mod.CGspace, bsz, sums)
    assert torch.equal(ff, y)
    # the kernel rounds |z| to float32 (its square root is within one ulp) and adds in float64
    mod_z = y.double().pow(2).sum(-1).sqrt()
    o, parts = 0, []
    for l, t in enumerate(int(v) for v in mod.t_FF):
        n = t * (2 * l + 1)
        parts.append(mod_z[:, o:o + n].reshape(bsz, t, 2 * l + 1))
        o += n
    s1, s2 = (torch.cat([(c ** k).sum((0, 2)) for c in parts]) for k in (1, 2))
    assert torch.allclose(sums[:, 0], s1, rtol=4e-7, atol=1e-12) and torch.allclose(sums[:, 1], s2, rtol=8e-7, atol=1e-12)


def test_large_batches_fit_the_static_statistics_area(dev):  # noqa: F811
    """The groups of the pair kernel grow with the batch; their partial statistics stay inside the fixed area wherever
    there is room for the task kernel's groups (29 of them here), at any batch."""
    from cgnet_amd import CG_layers, _lib
    lib = _lib.load()
    limit = int(lib.cgnet_sparse_forward_stats_static_limit())
    mod = CG_layers.CG_woFilter_cuda(8, [8, 7, 6, 8, 6, 8, 7, 5, 8], device=dev)
    plan = mod.native_plan()
    for bsz in (4, 31, 128, 1000, 4097, 1000003):
        assert 0 < lib.cgnet_sparse_forward_stats_workspace(plan._h, bsz) <= limit, bsz
    bsz = 8 * (limit // (16 * plan.sum_tFF)) + 13                      # eight samples a group would be too many groups
    g = torch.Generator(device=dev).manual_seed(8)
    x = torch.randn(bsz, plan.nF, 2, generator=g, device=dev)
    ff, ff_s = (torch.full((bsz, plan.nFF, 2), float("nan"), device=dev) for _ in range(2))
    sums, sums_s = (torch.full((plan.sum_tFF, 2), float("nan"), device=dev, dtype=torch.float64) for _ in range(2))
    plan.forward_stats(x, ff, mod.CGspace, bsz, sums)
    plan.forward_stats_static(x, ff_s, mod.CGspace, bsz, sums_s)
    assert torch.equal(ff, ff_s) and torch.equal(sums, sums_s)
    o = 0
    for l, t in enumerate(int(v) for v in mod.t_FF):                   # the last sample's and the sums of one degree's channels
        n = t * (2 * l + 1)
        if l == 5:
            z = ff[:, o:o + n].double().pow(2).sum(-1).sqrt().reshape(bsz, t, 2 * l + 1)
            c = int(sum(int(v) for v in mod.t_FF[:l]))
            assert torch.allclose(sums[c:c + t, 0], z.sum((0, 2)), rtol=4e-7, atol=1e-12)
        o += n
    alone = mod(x[-4:], straight_output=True)
    assert torch.equal(alone, ff[-4:])
