"""The backward organised by pairs of input degrees (cg_backward_pair_kernel) where its pieces have edges: tiles of whole rows and
of sixteen columns wherever they begin, a last tile that is short, one to three row tiles (and one row in the last), one to six
chunks of values of m, one to four groups of output degrees, a triple kept twice, empty degrees, units cut for small batches, work-groups
with samples left over; both sources of the product's gradient; and the rule that chooses the kernel.  Against the oracle the
tolerance of tests/test_gpu_parity.py: the strict bar, or three times what float32 arithmetic on the CPU is off by."""
import pytest
import torch

from tests.test_gpu_parity import (F32, assert_close, build_layer_pair, cg_oracle_fwd_bwd, check_layer_step, dev, edge_pairs,  # noqa: F401
                                   rand_straight, randn32)

pytestmark = pytest.mark.gpu

CASES = [
    # lmax, taus, B, triples
    (0, [3], 9, "default"),                                           # degree 0 alone: first and last channel of a sample in one tile
    (1, [1, 2], 1, "default"),
    (3, [2, 2, 2, 2], 33, "default"),                                 # eight work-groups of four samples and one sample more
    (4, [1, 13, 3, 16, 9], 5, "default"),                             # tiles of eight rows at most; sixteen columns of 13 and of 9
    (5, [12, 0, 7, 12, 1, 10], 6, "default"),                         # an empty degree; sixteen columns of 12 (three phases)
    (7, [5] * 8, 4, "mst"),                                           # fifteen values of m2: one row tile, full
    (8, [3, 1, 12, 4, 2, 6, 1, 12, 12], 3, "default"),                # seventeen: two, one row in the second
    (11, [12] * 12, 2, "default"),
    (13, [1] * 13 + [15], 7, "mst"),
    (15, [4, 16] * 8, 2, "default"),                                  # 31 values of m2, sixteen output degrees
    (16, [1, 2] * 8 + [3], 2, "default"),                             # 33: three row tiles, one row in the third; 17 degrees: cut, 16 and 1
    (20, [2] * 21, 1, "default"),                                     # 21 output degrees: cut, 16 and 5
    (23, [1, 2, 1] * 8, 3, "edge"),
    (3, [2, 3, 1, 2], 13, [[(1, 1)], [(1, 1), (2, 1), (2, 1)], [(2, 2), (2, 2), (3, 1)], [(3, 0)]]),   # kept twice
]


def _kernels(run):
    from cgnet_amd import _lib
    lib = _lib.load()
    lib.cgnet_profile_reset()
    lib.cgnet_profile_enable(1)
    run()
    torch.cuda.synchronize()
    lib.cgnet_profile_enable(0)
    return set(_lib.kernel_times())


def _module(dev, lmax, taus, mode):  # noqa: F811
    from cgnet_amd import CG_layers
    return CG_layers.CG_woFilter_cuda(lmax, taus, lll_mode=None if mode == "default" else edge_pairs(lmax) if mode == "edge" else mode,
                                      device=dev)


@pytest.mark.parametrize("lmax,taus,bsz,mode", CASES)
def test_pair_backward(dev, lmax, taus, bsz, mode):  # noqa: F811
    mod = _module(dev, lmax, taus, mode)
    plan = mod.native_plan()
    x64 = rand_straight(taus, bsz, seed=lmax + bsz)
    gy64 = randn32((bsz, plan.nFF, 2), torch.Generator().manual_seed(lmax))
    _, want = cg_oracle_fwd_bwd(lmax, taus, mod.lll_list, x64, gy64)
    _, twin = cg_oracle_fwd_bwd(lmax, taus, mod.lll_list, x64, gy64, dtype=F32)
    x, gy = x64.float().to(dev), gy64.float().to(dev)
    gx = torch.full_like(x, float("nan"))
    names = _kernels(lambda: plan.backward(x, gx, gy, mod.CGspace, bsz))
    assert names == {"pack_coef_back_kernel", "cg_backward_pair_kernel", "cg_backward_rows_kernel"}
    assert_close(gx, want, "pair backward", twin)


@pytest.mark.parametrize("lmax,taus,bsz,mode", [CASES[0], CASES[2], CASES[5], CASES[8], CASES[10]])
def test_non_finite_gradients_stay_in_their_sample(dev, lmax, taus, bsz, mode):  # noqa: F811
    """A load of sixteen bytes holds entries next to those it is for, at the ends of a sample too: never another sample's."""
    mod = _module(dev, lmax, taus, mode)
    plan = mod.native_plan()
    g = torch.Generator(device=dev).manual_seed(lmax)
    x, gy = (torch.randn(bsz, n, 2, generator=g, device=dev) for n in (plan.nF, plan.nFF))
    want = torch.empty_like(x)
    plan.backward(x, want, gy, mod.CGspace, bsz)
    bad = bsz // 2
    gy[bad, 0] = float("inf")
    gy[bad, -1] = float("nan")
    got = torch.empty_like(x)
    plan.backward(x, got, gy, mod.CGspace, bsz)
    others = torch.arange(bsz, device=dev) != bad
    assert torch.equal(got[others], want[others])
    assert not torch.isfinite(got[bad]).all()


@pytest.mark.parametrize("lmax,tin,tout,bsz,sparse", [
    (3, [2, 2, 2, 2], [2, 2, 2, 2], 4, False),
    (5, [12, 7, 5, 4, 4, 3], [12, 7, 5, 4, 4, 3], 9, False),         # falling channel counts: steps of zeros in the higher degrees
    (6, [3, 0, 16, 1, 9, 2, 4], [1, 5, 0, 16, 2, 3, 8], 6, True),     # no inputs, no outputs
    (9, [1] * 10, [4] * 10, 1, False),
    (16, [1] * 17, [2] * 17, 2, True),
    (20, [1] * 21, [1] * 21, 2, False),                               # pairs of up to 21 output degrees, cut after sixteen
])
def test_layer_backward_of_few_channels(dev, monkeypatch, lmax, tin, tout, bsz, sparse):  # noqa: F811
    """The one-kernel backward makes the product's gradient in the order of the gFF kernel and goes on as the stand-alone
    backward does: the same input gradient, bit for bit, as the two kernels; and both against the oracle."""
    mod, ora, twin, w64 = build_layer_pair(dev, lmax, tin, tout, sparse, True, seed=lmax)
    assert mod.native_layer_plan().fused_backward_supported
    x64 = rand_straight(tin, bsz, seed=7 * lmax)
    go = randn32((bsz, sum(t * (2 * l + 1) for l, t in enumerate(tout)), 2), torch.Generator().manual_seed(lmax)).float().to(dev)
    stds0 = mod.bnWMM.bn_stds.detach().clone()
    grads = []
    for one_kernel in (False, True):
        mod.fused_backward = one_kernel
        mod.bnWMM.bn_cnt = 1.
        with torch.no_grad():
            mod.bnWMM.bn_stds.copy_(stds0)
        mod.bnWMM.W.grad = None
        x = x64.float().to(dev).requires_grad_(True)
        out = mod(x, straight_output=True)
        names = _kernels(lambda: out.backward(go))
        assert "cg_backward_pair_kernel" in names and ("wmm_gradff_mfma_kernel" in names) != one_kernel
        grads.append((x.grad, mod.bnWMM.W.grad))
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])
    with torch.no_grad():
        mod.bnWMM.bn_stds.copy_(stds0)
    mod.bnWMM.bn_cnt = 1.
    check_layer_step(dev, mod, ora, twin, w64, x64, go.double().cpu())


@pytest.mark.parametrize("lmax,tau,batches", [(5, 16, (2, 40)), (8, 12, (3, 70)), (6, 7, (5, 200))])
def test_rule_and_other_kernels(dev, lmax, tau, batches):  # noqa: F811
    """Large batches of the reduced triples belong to the kernels that work triple by triple, stand-alone and (8..16 channels) inside
    the layer; a sample's gradient on either side of the rule differs by rounding."""
    from cgnet_amd import CG_layers
    taus = [tau] * (lmax + 1)
    mod = CG_layers.CGBN_cuda(lmax, taus, taus, sparse_flag=True, device=dev)
    mod.eval()
    g = torch.Generator(device=dev).manual_seed(lmax)
    few, many = batches
    x = torch.randn(many, mod.cg.native_plan().nF, 2, generator=g, device=dev)
    go = torch.randn(many, sum(tau * (2 * l + 1) for l in range(lmax + 1)), 2, generator=g, device=dev)
    for fused in (False, True):
        mod.fused_backward = fused
        got = []
        for n in (few, many):
            xs = x[:n].clone().requires_grad_(True)
            out = mod(xs, straight_output=True)
            names = _kernels(lambda: out.backward(go[:n].contiguous()))
            by_pairs = n == few or (fused and tau < 8)
            assert ("cg_backward_pair_kernel" in names) == by_pairs, (fused, n, names)
            got.append(xs.grad[:few])
        # sums of some thousand products of either order: the error of a sum grows like the root of its terms, and the largest
        # entry is a few times their root mean square
        assert (got[0] - got[1]).abs().max() <= 2e-5 * got[0].abs().max()
