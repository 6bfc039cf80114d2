"""Gradient of the product tensor as products of bfloat16 pieces: taken where every degree with output channels has thirteen to sixteen."""
import pytest
import torch

from tests.test_gpu_back_pairs import _kernels
from tests.test_gpu_parity import dev, rand_straight  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,t_ff,t_o,bsz,spread", [
    (0, [17], [13], 1, 0),                                  # one value of m, a tile of one channel
    (3, [64, 16, 65, 15], [13, 16, 14, 0], 5, 0),           # tiles of channels full and not, a degree without outputs
    (7, [40] * 8, [16] * 8, 3, 0),                          # 15 values of m: a column tile short of one
    (11, [33] * 12, [14, 0, 13, 15] * 3, 2, 0),             # the last degree of three column tiles
    (12, [18] * 12 + [65], [13] * 12 + [15], 3, 0),         # the first of four, in a kernel of its own
    (16, [3] * 15 + [80, 17], [16] * 17, 2, 0),             # 66 columns: the fifth tile has two
    (19, [1] * 18 + [64, 33], [13] * 20, 1, 60),            # 78 columns
    (23, [2] * 20 + [16, 48, 65, 20], [14] * 24, 2, 0),     # six column tiles
    (24, [20] * 25, [13] * 25, 1, 0),                       # seven: the fp32 instructions
    (3, [24] * 4, [13] * 4, 4, 60),                         # rows and columns of very different size
    (3, [24] * 4, [12] * 4, 4, 60),                         # twelve channels: the fp32 instructions
    (13, [24] * 14, [12] * 14, 2, 60),
])
def test_product_gradient(dev, lmax, t_ff, t_o, bsz, spread):  # noqa: F811
    g = torch.Generator().manual_seed(lmax + spread)
    w, go = [], []
    for l, (k, n) in enumerate(zip(t_ff, t_o)):
        m = 2 * l + 1
        w.append(torch.randn(n, k, 2, generator=g) * torch.exp2(torch.randint(-spread, spread + 1, (1, k, 1), generator=g).float()))
        go.append(torch.randn(bsz, n, m, 2, generator=g) * torch.exp2(torch.randint(-spread, spread + 1, (bsz, 1, m, 1), generator=g).float()))
    std = torch.rand(sum(t_ff), generator=g) + 0.5
    names = _check(dev, w, go, std)
    assert ("pack_w_gradff_split_kernel" in names) == (min(t for t in t_o if t) >= 13 and lmax <= 23)


def _gradient(dev, w, go, std):  # noqa: F811
    """Gradient of the product tensor, per degree [sample, channel, m], and the kernels of the backward."""
    from cgnet_amd import CG_layers
    bsz = go[0].shape[0]
    t_ff, t_o = [v.shape[1] for v in w], [v.shape[0] for v in w]
    mod = CG_layers.MyBatchNormWeightMM_cuda(len(w) - 1, t_ff, t_o)
    with torch.no_grad():
        mod.W.copy_(torch.cat([v.reshape(-1, 2) for v in w]))
        mod.bn_stds.copy_(std)
    mod.eval()
    x = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(t_ff)), 2, generator=torch.Generator().manual_seed(1)).to(dev).requires_grad_(True)
    out = mod(x)
    names = _kernels(lambda: out.backward(torch.cat([v.reshape(bsz, -1, 2) for v in go], 1).to(dev)))
    got, at = [], 0
    for l, k in enumerate(t_ff):
        got.append(x.grad[:, at:at + k * (2 * l + 1)].reshape(bsz, k, 2 * l + 1, 2).cpu())
        at += k * (2 * l + 1)
    return got, names


def _check(dev, w, go, std):  # noqa: F811
    got, names = _gradient(dev, w, go, std)
    cplx = lambda t: torch.view_as_complex(t.double().contiguous())  # noqa: E731
    at, err, all_terms = 0, 0., 0.
    for l, (have, v, h) in enumerate(zip(got, w, go)):
        n, k = v.shape[:2]
        have, h, v = cplx(have), cplx(h), cplx(v) / std[at:at + k].double().clamp_min(1e-5)
        want, terms = torch.einsum("ok,bom->bkm", v.conj(), h), torch.einsum("ok,bom->bkm", v.abs(), h.abs())
        # The division rounds a weight (2^-24), the products left out are at most 2^-23 of theirs, and 2 n products of six parts are added
        # in fp32: at most 2^-24 of the sum of their moduli an addition, whatever the order, of which the parts after the first weigh
        # 2^-7 in all; twice that for both parts.  No term in the largest entry of anything.
        bound = (2 ** -24 * (1 + 2 * n * (1 + 2 ** -7)) + 2 ** -23) * 2 * terms + 2. ** -148
        assert ((have - want).abs() <= bound).all(), l
        miss = ((have - want).abs() - 2. ** -149).clamp_min(0.)    # less the last place of a result that is not normal
        err += miss.square().div(terms.square().clamp_min(2. ** -200)).sum()
        all_terms += float(((want.abs() / terms.clamp_min(2. ** -100)) ** 2).sum())
        at += k
    # entries as exact as chains of fp32 products leave them, each in terms of its own size
    assert err ** 0.5 < 4e-7 * all_terms ** 0.5
    return names


def _inverse(n, decades):
    """Sizes of output channels in W, and their inverse in gO."""
    r = 10. ** (decades * (torch.arange(n) / max(1, n - 1) - 0.5))
    return r[torch.randperm(n, generator=torch.Generator().manual_seed(n))]


@pytest.mark.parametrize("decades", [0, 6, 10, 30])
def test_output_channels_of_different_scale(dev, decades):  # noqa: F811
    """An output channel that the next layer's stds divide by s sends back a gradient of 1 / s."""
    g = torch.Generator().manual_seed(decades)
    w, go = [], []
    for l, (k, n) in enumerate([(33, 14), (16, 16), (40, 13), (17, 15)]):
        r = _inverse(n, decades)
        w.append(torch.randn(n, k, 2, generator=g) * r[:, None, None])
        go.append(torch.randn(3, n, 2 * l + 1, 2, generator=g) / r[None, :, None, None])
    assert "pack_w_gradff_split_kernel" in _check(dev, w, go, torch.rand(106, generator=g) + 0.5)


@pytest.mark.parametrize("size_w,size_go", [(-62, -62), (-20, -100), (0, -140), (61, 61), (20, 100), (-100, 100), (100, -100)])
def test_sizes_of_both_operands(dev, size_w, size_go):  # noqa: F811
    """What is in range in the result is in range on the way.  (2^61 twice: 26 products of normal numbers stay below 2^6 of 2^122.)"""
    g = torch.Generator().manual_seed(5)
    w, go = [], []
    for l in range(3):
        w.append(torch.randn(13, 20, 2, generator=g) * 2. ** size_w)
        go.append((torch.randn(2, 13, 2 * l + 1, 2, generator=g).double() * 2. ** size_go).float())
    if size_go >= -100:                                     # one output channel of the opposite size, whose partner is zero
        for v in w:
            v[3] = 0.
        for h in go:
            h[:, 3] = 2. ** -size_go
            h[:, 7] = 0.
        w[1][7] = 2. ** -size_w
    assert "pack_w_gradff_split_kernel" in _check(dev, w, go, torch.ones(60))


def _draw(seed):
    g = torch.Generator().manual_seed(seed)
    sizes = [(33, 14), (16, 16), (80, 13), (17, 15)]
    return ([torch.randn(n, k, 2, generator=g) for k, n in sizes],
            [torch.randn(3, n, 2 * l + 1, 2, generator=g) for l, (_, n) in enumerate(sizes)])


def test_infinite_weights(dev):  # noqa: F811
    """A weight that is not finite gives what a chain of fp32 products gives, and nothing to other channels."""
    w, go = _draw(7)
    clean, _ = _gradient(dev, w, go, torch.ones(146))
    w[1][3, 4, 0] = float("inf")
    w[2][5, 70, 1] = -float("inf")
    w[3][0, 16, 0] = float("nan")
    got, names = _gradient(dev, w, go, torch.ones(146))
    assert "pack_w_gradff_split_kernel" in names
    signs = lambda t: torch.sign(t) * float("inf")  # noqa: E731
    assert torch.equal(got[1][:, 4], signs(go[1][:, 3]))   # conj(inf) (x + i y) = inf x + i inf y
    assert torch.equal(got[2][:, 70], signs(torch.stack([-go[2][:, 5, :, 1], go[2][:, 5, :, 0]], -1)))    # conj(-i inf) (x + i y)
    assert torch.isnan(got[3][:, 16]).all()
    for l, c in ((1, 4), (2, 70), (3, 16)):
        got[l][:, c] = clean[l][:, c]
    assert all(torch.equal(a, b) for a, b in zip(got, clean))


@pytest.mark.parametrize("lmax", [0, 2])
def test_infinite_weight_in_a_layer(dev, lmax):  # noqa: F811
    """The layer's kernel makes of it what the two kernels make: infinities where one degree is alone, and not finite is the same place."""
    from cgnet_amd import CG_layers
    taus = [9] * (lmax + 1)
    mod = CG_layers.CGBN_cuda(lmax, taus, [13] * (lmax + 1), device=dev)
    mod.eval()
    with torch.no_grad():
        mod.bnWMM.W[5, 0] = float("inf")
    go = torch.randn(2, 13 * (lmax + 1) ** 2, 2, generator=torch.Generator().manual_seed(1)).to(dev)
    grads = []
    for one_kernel in (False, True):
        mod.fused_backward = one_kernel
        x = rand_straight(taus, 2, seed=lmax).float().to(dev).requires_grad_(True)
        mod(x, straight_output=True).backward(go)
        grads.append(x.grad)
    if lmax == 0:
        assert torch.isinf(grads[1]).any()
        assert torch.equal(grads[0].nan_to_num(3., 1e38, -1e38), grads[1].nan_to_num(3., 1e38, -1e38))
    fine = torch.isfinite(grads[0])
    assert torch.equal(fine, torch.isfinite(grads[1])) and torch.equal(grads[0][fine], grads[1][fine])


@pytest.mark.parametrize("which", ["gO", "weights"])
def test_largest_numbers(dev, which):  # noqa: F811
    """The largest fp32 number rounds to infinity as a bfloat16."""
    w, go = _draw(8)
    largest = torch.finfo(torch.float32).max
    if which == "gO":
        go[2][1, 3, 2, 1] = -largest
        w[2] *= 0.01
    else:
        w[1][3, 4, 0] = largest
        go[1] *= 0.01
    _check(dev, w, go, torch.ones(146))


@pytest.mark.parametrize("decades", [0, 10])
@pytest.mark.parametrize("lmax,tin,tout,bsz,sparse", [
    (2, [3, 1, 2], [13, 13, 13], 1, False),
    (6, [16, 5, 9, 0, 2, 8, 12], [16, 14, 0, 13, 15, 13, 16], 5, False),
    (9, [4] * 10, [14] * 10, 3, True),
    (13, [9] * 14, [16] * 14, 2, False),
    (18, [2] * 19, [13] * 19, 1, False),
    (22, [1] * 23, [15] * 23, 1, False),
    (9, [4] * 10, [12] * 10, 3, True),                      # twelve: both on the fp32 instructions
])
def test_layer_makes_the_same_gradient(dev, lmax, tin, tout, bsz, sparse, decades):  # noqa: F811
    """Inside the layer and in the mixing's kernel the products are the same and are added in the same order."""
    from cgnet_amd import CG_layers
    torch.manual_seed(lmax)
    mod = CG_layers.CGBN_cuda(lmax, tin, tout, sparse_flag=sparse, device=dev)
    mod.eval()
    go = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(tout)), 2, generator=torch.Generator().manual_seed(1))
    at = wt = 0
    for l, (n, k) in enumerate(zip(tout, (int(t) for t in mod.t_FF))):
        r = _inverse(n, decades)
        go[:, at:at + n * (2 * l + 1)] /= r.repeat_interleave(2 * l + 1)[None, :, None]
        with torch.no_grad():
            mod.bnWMM.W[wt:wt + n * k] *= r.repeat_interleave(k)[:, None].to(dev)
        at, wt = at + n * (2 * l + 1), wt + n * k
    go = go.to(dev)
    grads = []
    for one_kernel in (False, True):
        mod.fused_backward = one_kernel
        x = rand_straight(tin, bsz, seed=lmax).float().to(dev).requires_grad_(True)
        out = mod(x, straight_output=True)
        names = _kernels(lambda: out.backward(go))
        assert "cg_backward_pair_kernel" in names and ("wmm_gradff_mfma_kernel" in names) != one_kernel
        grads.append(x.grad)
    assert torch.isfinite(grads[0]).all() and torch.equal(grads[0], grads[1])
