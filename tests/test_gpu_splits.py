"""Fragment norm + mixing where the rules that cut the work change: lengths of the forward's channel slices (32 to 256
channels), chunks of samples of the weight gradient, groups of samples of the product-tensor gradient."""
import pytest
import torch

from tests.test_gpu_parity import dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,t_ff,t_o,bsz", [
    (2, {0: 33, 1: 128, 2: 31}, {0: 3, 1: 17, 2: 1}, 1),          # one slice: splitting does not pay
    (2, {0: 33, 1: 129, 2: 32}, {0: 3, 1: 17, 2: 1}, 1),          # slices of 32: one channel over, exact
    (1, {0: 65, 1: 257}, {0: 4, 1: 4}, 9),                        # chunks of three samples, groups of two and a single one
    (6, {6: 2500, 3: 700}, {6: 5, 3: 20}, 130),                   # slices of 64, two row chunks
    (11, {11: 1100, 4: 900, 0: 0}, {11: 12, 4: 3, 0: 2}, 300),    # slices of 128 / 256, a degree with outputs only
    (24, {24: 40, 9: 300}, {24: 2, 9: 16}, 5),                    # more than three column tiles
])
def test_mixing_splits(dev, lmax, t_ff, t_o, bsz):  # noqa: F811
    from cgnet_amd import CG_layers
    t_ff = [t_ff.get(l, 0) for l in range(lmax + 1)]
    t_o = [t_o.get(l, 0) for l in range(lmax + 1)]
    mod = CG_layers.MyBatchNormWeightMM_cuda(lmax, t_ff, t_o)
    g = torch.Generator().manual_seed(lmax + bsz)
    ff = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(t_ff)), 2, generator=g)
    go = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(t_o)), 2, generator=g)
    w = torch.randn(mod.W.shape, generator=g)
    std = torch.rand(sum(t_ff), generator=g) + 0.5
    with torch.no_grad():
        mod.W.copy_(w)
        mod.bn_stds.copy_(std)
    mod.eval()
    x = ff.to(dev).requires_grad_(True)
    out = mod(x)
    out.backward(go.to(dev))
    offs = [0, 0, 0, 0]
    cplx = lambda t: torch.view_as_complex(t.double().contiguous())  # noqa: E731
    ff, go, w = cplx(ff), cplx(go), cplx(w)
    got = [cplx(t.detach().cpu()) for t in (out, x.grad, mod.W.grad)]
    for l, (k, n) in enumerate(zip(t_ff, t_o)):
        m = 2 * l + 1
        f = ff[:, offs[0]:offs[0] + k * m].reshape(bsz, k, m)
        h = go[:, offs[1]:offs[1] + n * m].reshape(bsz, n, m)
        v = w[offs[2]:offs[2] + k * n].reshape(n, k) / std[offs[3]:offs[3] + k]
        want = [torch.einsum("ok,bkm->bom", v, f), torch.einsum("ok,bom->bkm", v.conj(), h),
                torch.einsum("bom,bkm->ok", h, f.conj()) / std[offs[3]:offs[3] + k]]
        have = [got[0][:, offs[1]:offs[1] + n * m], got[1][:, offs[0]:offs[0] + k * m], got[2][offs[2]:offs[2] + k * n]]
        for a, b, terms in zip(have, want, (k, n, bsz * m)):
            if b.numel():
                # 2 terms real products are added in single precision: every addition rounds a partial sum, no larger
                # than the largest result, by half an ulp; the errors add up as a random walk, five sigma of it (a
                # channel, sample or slice left out would show as 1 / sqrt(terms))
                bound = 5 * 6e-8 * (2 * terms) ** 0.5 * b.abs().max()
                assert (a.reshape(b.shape) - b).abs().max() <= bound, (l, terms)
            else:
                assert a.abs().sum() == 0
        offs = [offs[0] + k * m, offs[1] + n * m, offs[2] + k * n, offs[3] + k]


@pytest.mark.parametrize("lmax,tau", [(3, 16), (8, 9), (11, 5)])
def test_workspace_of_a_batch_serves_smaller_ones(dev, lmax, tau):  # noqa: F811
    """Smaller batches take shorter slices, which leave more partial outputs a sample."""
    from cgnet_amd import CG_layers, CGutils, _lib
    pairs = CGutils.SparseLtuples.compute_default_ltuples(lmax)
    mod = CG_layers.MyBatchNormWeightMM_cuda(lmax, [len(p) * tau * tau for p in pairs], [tau] * (lmax + 1))
    plan = mod.native_plan()
    sizes = [_lib.load().cgnet_FN_WMM_forward_workspace(plan._h, b) for b in range(1, 400)]
    assert sizes == sorted(sizes) and sizes[0] > 0
