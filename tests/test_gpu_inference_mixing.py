"""Evaluation without the product tensor: every output entry is as exact as a chain of fp32 products, whatever the sizes beside it."""
import pytest
import torch

from tests.test_gpu_back_pairs import _kernels
from tests.test_gpu_parity import dev, rand_straight  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    (0, [8], [1], 1, False, 0),                             # one value of m, sixteen steps on four shares
    (3, [9, 11, 8, 10], [16, 12, 0, 3], 5, False, 0),       # last steps of every length, a degree without outputs
    (7, [16] * 8, [16] * 8, 3, False, 0),                   # one column tile, sixteen steps a share
    (8, [13] * 9, [9] * 9, 2, False, 0),                    # 17 values of m: two column tiles, shares of ten and eleven steps
    (15, [16] * 16, [16] * 16, 1, True, 0),
    (5, [12] * 6, [12] * 6, 4, False, 6),                   # channels, weights and stds of very different size
]


def _layer(lmax, tin, tout, bsz, sparse, spread, dev):  # noqa: F811
    from cgnet_amd import CG_layers
    g = torch.Generator().manual_seed(lmax + spread)
    mod = CG_layers.CGBN_cuda(lmax, tin, tout, sparse_flag=sparse, device=dev)
    std = torch.exp2(torch.rand(mod.bnWMM.bn_stds.shape, generator=g) * 2 * spread - spread)
    w = torch.randn(mod.bnWMM.W.shape, generator=g)
    with torch.no_grad():
        mod.bnWMM.W.copy_(w)
        mod.bnWMM.bn_stds.copy_(std)
    mod.eval()
    x = rand_straight(tin, bsz, seed=lmax).float()
    at = 0
    for l, t in enumerate(tin):
        scale = torch.exp2(torch.randint(-spread, spread + 1, (t,), generator=g).float())
        x[:, at:at + t * (2 * l + 1)] *= scale.repeat_interleave(2 * l + 1)[None, :, None]
        at += t * (2 * l + 1)
    return mod, w, std, x.to(dev)


def _parts(mod, product, w, std, tout):
    """Per degree: places of the product, of the outputs, and W / std (complex, 64 bits)."""
    fo = oo = wo = to = 0
    w, std = torch.view_as_complex(w.double().contiguous()), std.double().clamp_min(float(mod.bnWMM.bn_eps))
    for l, (k, n) in enumerate(zip([int(t) for t in product.t_FF], tout)):
        m = 2 * l + 1
        yield slice(fo, fo + k * m), slice(oo, oo + n * m), w[wo:wo + k * n].reshape(n, k) / std[to:to + k], m
        fo, oo, wo, to = fo + k * m, oo + n * m, wo + k * n, to + k


def _check(mod, w, std, x, tout, sparse):
    """Against the mixing of the product tensor in 64 bits, entry by entry; returns what the layer gave."""
    from cgnet_amd import CG_layers
    product = CG_layers.CG_woFilter_cuda(mod.lmax, [int(t) for t in mod.t_F], lll_mode="mst" if sparse else None)
    out = []
    with torch.no_grad():
        names = _kernels(lambda: out.append(mod(x, straight_output=True)))
        ff = product(x, straight_output=True)               # by the same steps: the tiles that were mixed
    assert "cgbn_forward_fused_kernel" in names
    cplx = lambda t: torch.view_as_complex(t.double().cpu().contiguous())  # noqa: E731
    got, ff, bsz = cplx(out[0]), cplx(ff), x.shape[0]
    for l, (fs, os, v, m) in enumerate(_parts(mod, product, w, std, tout)):
        n, k = v.shape
        if n == 0:
            continue
        z, have = ff[:, fs].reshape(bsz, k, m), got[:, os].reshape(bsz, n, m)
        want = torch.einsum("oc,bcm->bom", v, z)
        # The division rounds a weight (2^-24) and 2 k products are added in fp32: at most 2^-24 of the sum of their moduli an addition,
        # whatever the order; twice that for both parts.
        terms = torch.einsum("oc,bcm->bom", v.abs(), z.abs())
        assert ((have - want).abs() <= 2 ** -24 * (2 + 2 * k) * 2 * terms).all(), l
        # and as chains of fp32 products do at the least: the error over all, and that of every column m against the column's terms
        assert (have - want).abs().square().sum().sqrt() < 4e-7 * want.abs().square().sum().sqrt(), l
        err, size = (have - want).abs().square().sum((0, 1)).sqrt(), terms.square().sum((0, 1)).sqrt()
        assert (err <= 4e-7 * size).all(), (l, float((err / size.clamp_min(1e-300)).max()))
    return out[0]


@pytest.mark.parametrize("lmax,tin,tout,bsz,sparse,spread", CASES)
def test_mixing(dev, lmax, tin, tout, bsz, sparse, spread):  # noqa: F811
    mod, w, std, x = _layer(lmax, tin, tout, bsz, sparse, spread, dev)
    _check(mod, w, std, x, tout, sparse)


@pytest.mark.parametrize("kind", ["decades0", "decades4", "decades8", "dead", "zonal"])
def test_channels_of_different_scale(dev, kind):  # noqa: F811
    """Channels spread over decades with stds that follow them, channels that are dead with stds at eps, fragments that nearly vanish
    off m = 0: evaluation answers as through the product tensor, which training takes."""
    from cgnet_amd import CG_layers
    lmax, tau, bsz = 8, 12, 3
    mod, w, std, x = _layer(lmax, [tau] * (lmax + 1), [tau] * (lmax + 1), bsz, False, 0, dev)
    product = CG_layers.CG_woFilter_cuda(lmax, [tau] * (lmax + 1))
    at = 0
    for l in range(lmax + 1):
        part = x[:, at:at + tau * (2 * l + 1)].reshape(bsz, tau, 2 * l + 1, 2)
        if kind.startswith("decades"):                      # of the product's channels
            part *= (100. * 10. ** (-int(kind[7:]) / 2. * torch.arange(tau, device=dev) / (tau - 1)))[None, :, None, None]
        elif kind == "dead":
            part *= 30.
            part[:, ::4] = 0.
        else:
            part[:, :, torch.arange(2 * l + 1) != l] *= 1e-8
        at += tau * (2 * l + 1)
    if kind != "zonal":
        with torch.no_grad():
            ff = product(x, straight_output=True).double().cpu()
        std, at = [], 0
        for l, k in enumerate(int(t) for t in product.t_FF):
            std.append(ff[:, at:at + k * (2 * l + 1)].reshape(bsz, k, 2 * l + 1, 2).square().sum(3).mean((0, 2)).sqrt())
            at += k * (2 * l + 1)
        std = torch.cat(std).float()
        with torch.no_grad():
            mod.bnWMM.bn_stds.copy_(std)
    out = _check(mod, w, std, x, [tau] * (lmax + 1), False)
    with torch.no_grad():
        mod.fused_inference = False
        through_ff = mod(x, straight_output=True)
    # two roundings of the same chains (test_mixing's bound for each); zonal columns of nearly nothing count for themselves
    assert (out - through_ff).norm() <= 8e-7 * through_ff.norm()
    at = 0
    for l in range(lmax + 1):
        a, b = (t[:, at:at + tau * (2 * l + 1)].double().reshape(bsz, tau, 2 * l + 1, 2) for t in (out, through_ff))
        assert ((a - b).square().sum((0, 1, 3)).sqrt() <= 2e-6 * b.square().sum((0, 1, 3)).sqrt()).all(), l
        at += tau * (2 * l + 1)


def test_infinite_weight_stays_where_it_is(dev):  # noqa: F811
    mod, w, _, x = _layer(3, [9] * 4, [10] * 4, 2, False, 0, dev)
    with torch.no_grad():
        clean = mod(x, straight_output=True)
        mod.bnWMM.W[17, 0] = float("inf")
        mod.bnWMM.W[int(mod.bnWMM.W.shape[0]) - 3, 1] = float("nan")
        out = mod(x, straight_output=True)
        mod.fused_inference = False
        through_ff = mod(x, straight_output=True)
    finite = torch.isfinite(through_ff)
    assert not finite.all() and finite.any()
    assert torch.equal(torch.isfinite(out), finite) and torch.equal(out[finite], clean[finite])
    assert torch.equal(torch.isnan(out), torch.isnan(through_ff))


def test_infinite_entry_stays_in_its_sample(dev):  # noqa: F811
    """What is finite through the product tensor is finite here."""
    mod, _, _, x = _layer(6, [10] * 7, [9] * 7, 3, True, 0, dev)   # the last degree's entries of outermost m reach only some m
    with torch.no_grad():
        clean = mod(x, straight_output=True)
        x[1, 477, 0] = float("inf")
        x[2, 489, 1] = float("nan")
        out = mod(x, straight_output=True)
        mod.fused_inference = False
        through_ff = mod(x, straight_output=True)
    assert torch.equal(out[0], clean[0])
    finite = torch.isfinite(through_ff)
    assert not finite[1:].all() and finite[1:].any()
    assert torch.equal(torch.isfinite(out), finite)
    assert (out - through_ff)[finite].abs().max() <= 1e-5 * through_ff[finite].abs().max()
