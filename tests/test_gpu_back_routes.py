"""The backward goes by pairs of input degrees up to a batch, triple by triple above it, and cuts its work finer for small batches:
what a caller sees of that besides the results."""
import ctypes

import pytest
import torch

from tests import test_gpu_parity as parity
from tests.test_gpu_back_pairs import _kernels
from tests.test_gpu_parity import dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,tau,sparse", [
    (11, 12, False),                                       # by pairs throughout, three cuts
    (20, 3, False),
    (8, 12, True),                                         # pairs, then triples
    (11, 5, True),
    (15, 16, True),
])
def test_buffers_of_a_batch_serve_smaller_ones(dev, lmax, tau, sparse):  # noqa: F811
    """A caller allocates for its full batch and passes a shorter last one: sizes never fall with the batch, and a call on a small
    batch takes the buffers of a large one."""
    from cgnet_amd import CG_layers, _lib
    taus = [tau] * (lmax + 1)
    mod = CG_layers.CGBN_cuda(lmax, taus, [2] * (lmax + 1), sparse_flag=sparse, device=dev)
    lib, lp = _lib.load(), mod.native_layer_plan()
    cg = lp.cg_plan
    queries = {"backward": (lib.cgnet_sparse_backward_workspace, cg._h), "saved": (lib.cgnet_CGBN_saved_bytes, lp._h),
               "layer backward": (lib.cgnet_CGBN_backward_fused_workspace, lp._h)}
    batches = range(1, 260)
    sizes = {name: [query(plan, b) for b in batches] for name, (query, plan) in queries.items()}
    for name, got in sizes.items():
        assert got[0] > 0 and got == sorted(got), name
    big = {name: torch.empty(got[-1], dtype=torch.uint8, device=dev) for name, got in sizes.items()}
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    s = torch.cuda.current_stream(dev).cuda_stream
    ffs = torch.empty(30, cg.nFF, 2, device=dev)
    g = torch.Generator(device=dev).manual_seed(lmax)
    for b in (1, 19, 30):
        x, out = torch.randn(b, cg.nF, 2, generator=g, device=dev), torch.empty(b, lp.wmm_plan.nO, 2, device=dev)
        go, gff = torch.randn(out.shape, generator=g, device=dev), torch.randn(b, cg.nFF, 2, generator=g, device=dev)
        want, got = torch.empty_like(x), torch.empty_like(x)
        cg.backward(x, want, gff, mod.cg.CGspace, b)
        _lib.check(lib.cgnet_sparse_backward(cg._h, ptr(x), ptr(got), ptr(gff), ptr(mod.cg.CGspace), b, ptr(big["backward"]),
                                             big["backward"].numel(), s))
        assert torch.equal(got, want)
        args = mod.bnWMM.W.detach(), mod.cg.CGspace, b, mod.bnWMM.bn_stds, 1., 1e-5, _lib.FN_BATCHNORM
        own = lp.forward(x, ffs[:b], out, *args)
        lp.backward_fused(x, want, go, mod.bnWMM.W.detach(), mod.cg.CGspace, b, mod.bnWMM.bn_stds, 1e-5, _lib.FN_BATCHNORM, own)
        ws = torch.empty(lib.cgnet_CGBN_forward_workspace(lp._h, b), dtype=torch.uint8, device=dev)
        _lib.check(lib.cgnet_CGBN_forward(lp._h, ptr(x), ptr(ffs), ptr(out), ptr(mod.bnWMM.W), ptr(mod.cg.CGspace), b,
                                          ptr(mod.bnWMM.bn_stds), 1., 1e-5, _lib.FN_BATCHNORM, ptr(big["saved"]),
                                          big["saved"].numel(), ptr(ws), ws.numel(), s))
        _lib.check(lib.cgnet_CGBN_backward_fused(lp._h, None, ptr(got), ptr(go), None, None, b, None, 1e-5, _lib.FN_BATCHNORM,
                                                 ptr(big["saved"]), big["saved"].numel(), ptr(big["layer backward"]),
                                                 big["layer backward"].numel(), s))
        assert torch.equal(got, want)


@pytest.mark.parametrize("tau", [3, 9])
def test_layer_without_outputs(dev, tau):  # noqa: F811
    """No output channel in any degree: the output is empty (and lies nowhere), the gradients are zeros."""
    from cgnet_amd import CG_layers
    mod = CG_layers.CGBN_cuda(2, [tau] * 3, [0] * 3, device=dev)
    x = torch.randn(4, tau * 9, 2, device=dev, requires_grad=True)
    out = mod(x, straight_output=True)
    assert out.shape == (4, 0, 2)
    out.backward(torch.empty_like(out))
    assert x.grad.shape == x.shape and not x.grad.any()


# The kernels that work triple by triple serve the large batches of reduced triples; with CGNET_BWD_PAIRS=0 at plan creation they take
# the small batches that the oracle can follow too.
PRODUCTS = ([c for c in parity.CG_CASES if max(c[1]) <= 16] + parity._random_matrix_core_cases(12, 5) +
            parity._random_matrix_core_cases_high(6, 9) + [c for c in parity._random_cg_cases(24, 11) if max(c[1]) <= 16] +
            [(13, [16] * 14, 2, "mst"), (20, [9] * 21, 1, "mst"), (18, [8, 13, 16] * 6 + [10], 1, "mst"), (20, [3] * 21, 2, "mst")])


@pytest.mark.parametrize("lmax,taus,bsz,mode", PRODUCTS)
def test_product_triple_by_triple(dev, monkeypatch, lmax, taus, bsz, mode):  # noqa: F811
    """Ragged channels, row blocks cut by the LDS, partial last steps, one to three column tiles, empty degrees, against the oracle."""
    monkeypatch.setenv("CGNET_BWD_PAIRS", "0")
    names = _kernels(lambda: parity.test_cg_forward_backward(dev, lmax, taus, bsz, mode))
    matrix = all(t == 0 or 8 <= t <= 16 for t in taus)
    backward = {n for n in names if n in ("cg_backward_hybrid_kernel", "cg_backward_unit_kernel", "cg_backward_pair_kernel")}
    assert backward == {"cg_backward_hybrid_kernel" if matrix else "cg_backward_unit_kernel"}, names


@pytest.mark.parametrize("lmax,tin,tout,bsz,sparse,bn", parity.LAYER_CASES)
def test_layer_triple_by_triple(dev, monkeypatch, lmax, tin, tout, bsz, sparse, bn):  # noqa: F811
    monkeypatch.setenv("CGNET_BWD_PAIRS", "0")
    names = _kernels(lambda: parity.test_layer_forward_backward(dev, lmax, tin, tout, bsz, sparse, bn, "fused_backward"))
    one = all(t == 0 or 8 <= t <= 16 for t in tin) and max(tout) <= 16
    assert "cg_backward_pair_kernel" not in names and ("cgbn_backward_fused_kernel" in names) == one, names


def test_reason_of_a_layer_that_is_taken(dev, monkeypatch):  # noqa: F811
    """A layer that only the kernel by triples takes has no reason why it is not taken; one that neither takes has."""
    from cgnet_amd import CG_layers
    monkeypatch.setenv("CGNET_BWD_PAIRS", "0")
    for tau, taken in ((9, True), (3, False)):
        lp = CG_layers.CGBN_cuda(2, [tau] * 3, [2] * 3, device=dev).native_layer_plan()
        assert lp.fused_backward_supported == taken and bool(lp.fused_backward_reason) != taken


@pytest.mark.parametrize("test", [parity.test_invalid_table_slots_are_never_used, parity.test_fused_backward_builds_its_own_operands,
                                  parity.test_layer_steps_back_to_back])
def test_layer_properties_triple_by_triple(dev, monkeypatch, test):  # noqa: F811
    """The masked tables, the operands a backward makes itself, steps without a wait between them: as for the pairs."""
    monkeypatch.setenv("CGNET_BWD_PAIRS", "0")
    names = _kernels(lambda: test(dev))
    assert "cgbn_backward_fused_kernel" in names and "cg_backward_pair_kernel" not in names, names


@pytest.mark.parametrize("lmax,tau,sparse", [(15, 16, True), (8, 12, True), (11, 5, True), (11, 12, False)])
def test_occupancy_covers_every_kernel_of_a_plan(dev, monkeypatch, lmax, tau, sparse):  # noqa: F811
    """What a caller schedules by holds for each kernel the plan may launch."""
    from cgnet_amd import CG_layers
    make = lambda: CG_layers.CG_woFilter_cuda(lmax, [tau] * (lmax + 1), lll_mode="mst" if sparse else None, device=dev).native_plan()  # noqa: E731
    plan = make()
    monkeypatch.setenv("CGNET_BWD_PAIRS", "0")
    triples = make()
    assert triples.backward_groups >= 1 and plan.backward_groups * plan.backward_lds <= 160 * 1024
    if sparse:                                             # small batches by pairs, large ones triple by triple
        assert plan.backward_groups * plan.backward_lds >= triples.backward_groups * triples.backward_lds


@pytest.mark.parametrize("lmax,tau", [(20, 3), (20, 9), (20, 13), (21, 5), (23, 4), (23, 10), (23, 11), (23, 16)])
def test_two_groups_share_a_compute_unit(dev, lmax, tau):  # noqa: F811
    """The LDS of the pair kernel, whatever number of rows t1 its tiles touch; and the layout that this takes, against the oracle:
    a row of zeros between the sums and the fragments, one buffer of fragments where no unit has a second tile."""
    from cgnet_amd import CG_layers
    taus = [tau] * (lmax + 1)
    plan = CG_layers.CG_woFilter_cuda(lmax, taus, device=dev).native_plan()
    assert plan.backward_groups == 2 and 2 * plan.backward_lds <= 160 * 1024
    names = _kernels(lambda: parity.test_cg_forward_backward(dev, lmax, taus, 2 if tau < 10 else 1, "debug"))
    assert "cg_backward_pair_kernel" in names


@pytest.mark.parametrize("lmax,tau,sparse,layer,most", [
    (10, 12, False, False, 33),                            # by pairs 1.25 times as long at 64 samples
    (5, 7, False, False, 48),                              # 1.17 at 64
    (8, 14, True, False, 9),                               # 2.5 at 128
    (14, 10, True, True, 25),                              # 1.34 at 40
    (12, 15, True, True, 11),                              # 1.12 at 16
    (11, 12, False, True, None),                           # 0.76 at 128: every batch
    (11, 5, False, False, None),                           # 0.75 at 128
    (15, 16, False, False, None),
    (13, 16, True, True, None),
])
def test_largest_batch_by_pairs(dev, lmax, tau, sparse, layer, most):  # noqa: F811
    """The rule that leaves large batches to the kernels that work triple by triple, where those are the faster ones."""
    from cgnet_amd import CG_layers
    taus = [tau] * (lmax + 1)
    mod = CG_layers.CGBN_cuda(lmax, taus, [1] * (lmax + 1), sparse_flag=sparse, device=dev)
    plan, lp = mod.cg.native_plan(), mod.native_layer_plan()
    for bsz in (1, most, most + 1) if most else (1, 70):
        x = torch.randn(bsz, plan.nF, 2, device=dev)
        gx = torch.empty_like(x)
        if layer:
            go = torch.randn(bsz, lp.wmm_plan.nO, 2, device=dev)
            names = _kernels(lambda: lp.backward_fused(x, gx, go, mod.bnWMM.W.detach(), mod.cg.CGspace, bsz, None, 1e-5, 0))
        else:
            gff = torch.zeros(bsz, plan.nFF, 2, device=dev)
            names = _kernels(lambda: plan.backward(x, gx, gff, mod.cg.CGspace, bsz))
        assert ("cg_backward_pair_kernel" in names) == (not most or bsz <= most), (bsz, names)


@pytest.mark.parametrize("lmax,tau,tout,bsz", [(8, 12, 13, 70), (6, 9, 16, 60)])
@pytest.mark.parametrize("fold", [None, "0"])
def test_triples_beside_two_kernels(dev, monkeypatch, lmax, tau, tout, bsz, fold):  # noqa: F811
    """A layer of thirteen output channels and more, reduced triples, a batch past the rule, nothing switched: the layer's kernel makes the
    product's gradient on the fp32 instructions, the two kernels in bfloat16 pieces.  Each is as exact as chains of fp32 products, with
    the fold of the diagonal triples and without."""
    from cgnet_amd import CG_layers
    if fold:
        monkeypatch.setenv("CGNET_DIAG_FOLD", fold)
    mod = CG_layers.CGBN_cuda(lmax, [tau] * (lmax + 1), [tout] * (lmax + 1), sparse_flag=True, device=dev)
    mod.eval()
    g = torch.Generator(device=dev).manual_seed(lmax)
    x = torch.randn(bsz, mod.cg.native_plan().nF, 2, generator=g, device=dev)
    go = torch.randn(bsz, tout * (lmax + 1) ** 2, 2, generator=g, device=dev)
    grads = []
    for one_kernel in (True, False):
        mod.fused_backward = one_kernel
        xs = x.clone().requires_grad_(True)
        out = mod(xs, straight_output=True)
        names = _kernels(lambda: out.backward(go))
        assert "cg_backward_pair_kernel" not in names
        assert {"cgbn_backward_fused_kernel"} <= names if one_kernel else {"wmm_gradff_mfma_kernel", "pack_w_gradff_split_kernel"} <= names
        grads.append(xs.grad)
    # two roundings of the same sums: 2 tout products of a part each, then some hundred of those with fragments and coefficients; in terms
    # of the root mean square sqrt(n) 2^-24 each, and the largest difference a few times that
    diff, size = (grads[0] - grads[1]).double(), grads[0].double()
    assert diff.norm() <= 2e-6 * size.norm() and diff.abs().max() <= 2e-5 * size.abs().max()


def _reached(plan, l, m, channel=None):
    """Entries of F whose gradient holds entry m of degree l of the product's gradient: of one of its channels, or of all."""
    from cgnet_amd import CGutils
    n1 = plan.lmax + 1
    at = [0]
    for d in range(n1):
        at.append(at[-1] + plan.t_F[d] * (2 * d + 1))
    hit = torch.zeros(plan.nF, dtype=torch.bool)
    for (out, l1, l2), first in zip(CGutils.SparseLtuples.get_iter(plan.lmax, plan.llls), plan.t_offsets):
        t1, t2 = plan.t_F[l1], plan.t_F[l2]
        if out != l or not t1 * t2 or (channel is not None and not first <= channel < first + t1 * t2):
            continue
        a, b = (slice(None),) * 2 if channel is None else divmod(channel - first, t2)
        lo, hi = max(-l1, m - l2), min(l1, m + l2)
        hit[at[l1]:at[l1 + 1]].view(t1, -1)[a, l1 + lo:l1 + hi + 1] = True
        hit[at[l2]:at[l2 + 1]].view(t2, -1)[b, l2 + m - hi:l2 + m - lo + 1] = True
    return hit


def _places(width):
    """(degree, m, channel, entry): the ends of every degree, and some between."""
    begin = 0
    for l, t in enumerate(width):
        n = t * (2 * l + 1)
        for e in sorted({0, 2 * l, n // 3, n - 1}) if n else ():
            yield l, e % (2 * l + 1) - l, e // (2 * l + 1), begin + e
        begin += n


def _reached_by_fragment(plan, l, m):
    """Entries of F whose gradient holds entry m of a channel of degree l of F: for one of degree l1 all channels of l2 and the reverse."""
    from cgnet_amd import CGutils
    n1 = plan.lmax + 1
    at = [0]
    for d in range(n1):
        at.append(at[-1] + plan.t_F[d] * (2 * d + 1))
    hit = torch.zeros(plan.nF, dtype=torch.bool)
    for out, l1, l2 in CGutils.SparseLtuples.get_iter(plan.lmax, plan.llls):
        for here, other in ((l1, l2), (l2, l1)):
            if here == l and plan.t_F[l1] * plan.t_F[l2]:
                lo, hi = max(-other, -out - m), min(other, out - m)
                hit[at[other]:at[other + 1]].view(plan.t_F[other], -1)[:, other + lo:other + hi + 1] = True
    return hit


NOT_FINITE = [
    (0, [3], False),
    (1, [1, 2], False),
    (3, [2] * 4, False),
    (5, [12, 0, 7, 12, 1, 10], False),
    (9, [3] * 10, True),
    (11, [12] * 12, False),                                # tiles that begin inside a row
    (15, [4, 16] * 8, False),
    (20, [2] * 21, True),
]


@pytest.mark.parametrize("lmax,taus,sparse", NOT_FINITE)
def test_entries_that_are_not_finite_reach_what_depends_on_them(dev, lmax, taus, sparse):  # noqa: F811
    """Zero coefficients stand for no value of m, no degree and no channel, and zero times infinity is no zero: an infinity or NaN in
    the gradient that comes in changes the gradients it is a term of, and no other entry of its sample or of the batch."""
    from cgnet_amd import CG_layers
    mod = CG_layers.CGBN_cuda(lmax, taus, [2] * (lmax + 1), sparse_flag=sparse, device=dev).eval()
    plan, lp = mod.cg.native_plan(), mod.native_layer_plan()
    g = torch.Generator().manual_seed(lmax)
    with torch.no_grad():
        mod.bnWMM.W.copy_(torch.randn(mod.bnWMM.W.shape, generator=g))
        mod.bnWMM.bn_stds.fill_(1.)
    x = torch.randn(3, plan.nF, 2, generator=g).to(dev)

    for width, n, of_channel in ((plan.t_FF, plan.nFF, True), ([2] * (lmax + 1), lp.wmm_plan.nO, False)):
        gy = torch.randn(3, n, 2, generator=g).to(dev)
        want, got = torch.empty_like(x), torch.empty_like(x)

        def backward(grad):
            if of_channel:
                plan.backward(x, grad, gy, mod.cg.CGspace, 3)
            else:
                lp.backward_fused(x, grad, gy, mod.bnWMM.W.detach(), mod.cg.CGspace, 3, mod.bnWMM.bn_stds.data, 1e-5, 1)
        names = _kernels(lambda: backward(want))
        assert "cg_backward_pair_kernel" in names
        for k, (l, m, channel, entry) in enumerate(_places(width)):
            keep = gy[1, entry].clone()
            gy[1, entry, k % 2] = (float("inf"), float("nan"), -float("inf"))[k % 3]
            backward(got)
            gy[1, entry] = keep
            hit = torch.zeros(3, plan.nF, dtype=torch.bool)
            hit[1] = _reached(plan, l, m, channel if of_channel else None)
            assert torch.equal((~torch.isfinite(got)).any(-1).cpu(), hit), (of_channel, l, m, channel)
            assert torch.equal(got[0], want[0]) and torch.equal(got[2], want[2])
            # entries that a zero times infinity had reached are added up again, term by term: some thousand products in another
            # order, an error that grows like the root of the terms, and the largest entry a few times their root mean square
            rest = ~hit[1].to(dev)
            assert (got[1] - want[1])[rest].abs().sum() == 0 or (got[1] - want[1])[rest].abs().max() <= 2e-5 * want.abs().max()


@pytest.mark.parametrize("lmax,taus,sparse", NOT_FINITE)
def test_fragments_that_are_not_finite_reach_what_depends_on_them(dev, lmax, taus, sparse):  # noqa: F811
    from cgnet_amd import CG_layers
    mod = CG_layers.CGBN_cuda(lmax, taus, [2] * (lmax + 1), sparse_flag=sparse, device=dev).eval()
    plan, lp = mod.cg.native_plan(), mod.native_layer_plan()
    g = torch.Generator().manual_seed(lmax)
    x, gff, go = (torch.randn(3, n, 2, generator=g).to(dev) for n in (plan.nF, plan.nFF, lp.wmm_plan.nO))
    for backward in (lambda x, grad: plan.backward(x, grad, gff, mod.cg.CGspace, 3),
                     lambda x, grad: lp.backward_fused(x, grad, go, mod.bnWMM.W.detach(), mod.cg.CGspace, 3, None, 1e-5, 0)):
        want, got = torch.empty_like(x), torch.empty_like(x)
        backward(x, want)
        for k, (l, m, _, entry) in enumerate(_places(plan.t_F)):
            bad = x.clone()
            bad[1, entry, k % 2] = (float("inf"), float("nan"), -float("inf"))[k % 3]
            backward(bad, got)
            hit = torch.zeros(3, plan.nF, dtype=torch.bool)
            hit[1] = _reached_by_fragment(plan, l, m)
            finite = torch.isfinite(got).all(-1).cpu()
            assert not (~finite & ~hit).any() and torch.equal(got[0], want[0]) and torch.equal(got[2], want[2])
            assert not (finite & hit).any(), (l, m)


def test_time_of_a_gradient_with_one_infinity(dev):  # noqa: F811
    """It is a backward like others: adding up anew what the infinity had spoilt once took 600 times as long (lmax 20, 16 channels)."""
    from cgnet_amd import CG_layers
    mod = CG_layers.CGBN_cuda(20, [16] * 21, [16] * 21, device=dev).eval()
    plan, lp = mod.cg.native_plan(), mod.native_layer_plan()
    x, gff, go = (torch.randn(4, n, 2, device=dev) for n in (plan.nF, plan.nFF, lp.wmm_plan.nO))
    grad = torch.empty_like(x)
    for gy, backward in ((gff, lambda: plan.backward(x, grad, gff, mod.cg.CGspace, 4)),
                         (go, lambda: lp.backward_fused(x, grad, go, mod.bnWMM.W.detach(), mod.cg.CGspace, 4, None, 1e-5, 0))):
        times = []
        for value in (0., 0., float("inf")):                       # (the first call is a warm-up)
            gy[1, -1, 0] = value
            ends = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            ends[0].record()
            backward()
            ends[1].record()
            ends[1].synchronize()
            times.append(ends[0].elapsed_time(ends[1]))
        assert times[2] < 4 * times[1] + 5, times
