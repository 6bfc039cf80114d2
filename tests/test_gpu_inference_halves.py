"""Evaluation without the product tensor: the tile is mixed as products of halves, by the fp32 instructions where it is not finite."""
import pytest
import torch

from tests.test_gpu_back_pairs import _kernels
from tests.test_gpu_parity import dev, rand_straight  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [
    (0, [8], [1], 1, False, 0),                             # one value of m, two whole steps of 32 channels
    (3, [9, 11, 8, 10], [16, 12, 0, 3], 5, False, 0),       # last steps of every length, a degree without outputs
    (7, [16] * 8, [16] * 8, 3, False, 0),                   # one column tile: eight steps on seven shares
    (8, [13] * 9, [9] * 9, 2, False, 0),                    # 17 values of m: two column tiles, two steps on some of four shares
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


@pytest.mark.parametrize("lmax,tin,tout,bsz,sparse,spread", CASES)
def test_mixing(dev, lmax, tin, tout, bsz, sparse, spread):  # noqa: F811
    from cgnet_amd import CG_layers
    mod, w, std, x = _layer(lmax, tin, tout, bsz, sparse, spread, dev)
    product = CG_layers.CG_woFilter_cuda(lmax, tin, lll_mode="mst" if sparse else None)
    out = []
    with torch.no_grad():
        names = _kernels(lambda: out.append(mod(x, straight_output=True)))
        ff = product(x, straight_output=True)               # by the same steps: the tiles that were mixed
    assert "cgbn_forward_fused_kernel" in names
    cplx = lambda t: torch.view_as_complex(t.double().cpu().contiguous())  # noqa: E731
    got, ff, w, std = cplx(out[0]), cplx(ff), cplx(w), std.double()
    fo = oo = wo = to = 0
    for l, (k, n) in enumerate(zip([int(t) for t in product.t_FF], tout)):
        m = 2 * l + 1
        z = ff[:, fo:fo + k * m].reshape(bsz, k, m)
        v = w[wo:wo + k * n].reshape(n, k) / std[to:to + k]
        have, want = got[:, oo:oo + n * m].reshape(bsz, n, m), torch.einsum("oc,bcm->bom", v, z)
        # The division rounds a weight (2^-24), two pieces each factor (2^-23 of it, or 2^-39 of the largest of its tile or share), and
        # 2 k products are added in fp32: at most 2^-24 of the sum of their moduli an addition, whatever the order.
        terms = torch.einsum("oc,bcm->bom", v.abs(), z.abs())
        if n:
            largest = (v.abs().sum(1)[None] * z.abs().amax((1, 2))[:, None] + v.abs().max() * z.abs().sum(1).amax(1)[:, None])[..., None]
            assert ((have - want).abs() <= (2 ** -24 * (1 + 2 * k) + 2 ** -22) * 2 * terms + 2. ** -38 * 2 * largest).all(), l
            # and as chains of fp32 products do at the least
            err = ((have - want).abs().square().sum() / want.abs().square().sum()).sqrt()
            assert err < 4e-7, (l, float(err))
        fo, oo, wo, to = fo + k * m, oo + n * m, wo + k * n, to + k


def test_infinite_entry_stays_in_its_sample(dev):  # noqa: F811
    """A tile that holds an infinity takes the fp32 instructions: what is finite through the product tensor is finite here."""
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
