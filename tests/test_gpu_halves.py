"""Gradient of the product tensor as products of halves: taken where every degree with output channels has nine to sixteen."""
import pytest
import torch

from tests.test_gpu_back_pairs import _kernels
from tests.test_gpu_parity import dev, rand_straight  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,t_ff,t_o,bsz,spread", [
    (0, [17], [9], 1, 0),                                   # one value of m, a tile of one channel
    (3, [64, 16, 65, 15], [9, 16, 12, 0], 5, 0),            # tiles of channels full and not, a degree without outputs
    (7, [40] * 8, [16] * 8, 3, 0),                          # 15 values of m: a column tile short of one
    (11, [33] * 12, [12, 0, 13, 9] * 3, 2, 0),
    (24, [20] * 25, [10] * 25, 1, 0),                       # more than three column tiles
    (3, [24] * 4, [9] * 4, 4, 60),                          # rows and columns of very different size
    (3, [24] * 4, [8] * 4, 4, 60),                          # eight channels: the fp32 instructions
])
def test_product_gradient(dev, lmax, t_ff, t_o, bsz, spread):  # noqa: F811
    from cgnet_amd import CG_layers
    mod = CG_layers.MyBatchNormWeightMM_cuda(lmax, t_ff, t_o)
    g = torch.Generator().manual_seed(lmax + spread)
    offs = [0, 0, 0, 0]
    w = torch.randn(mod.W.shape, generator=g)
    std = torch.rand(sum(t_ff), generator=g) + 0.5
    rows = []
    for l, (k, n) in enumerate(zip(t_ff, t_o)):
        m = 2 * l + 1
        scale = torch.exp2(torch.randint(-spread, spread + 1, (bsz, 1, m, 1), generator=g).float())
        rows.append((torch.randn(bsz, n, m, 2, generator=g) * scale).reshape(bsz, n * m, 2))
        if n:
            part = w[offs[2]:offs[2] + k * n].reshape(n, k, 2)
            part *= torch.exp2(torch.randint(-spread, spread + 1, (1, k, 1), generator=g).float())
        offs[2] += k * n
    go = torch.cat(rows, 1)
    with torch.no_grad():
        mod.W.copy_(w)
        mod.bn_stds.copy_(std)
    mod.eval()
    x = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(t_ff)), 2, generator=g).to(dev).requires_grad_(True)
    out = mod(x)
    names = _kernels(lambda: out.backward(go.to(dev)))
    assert ("pack_w_gradff_split_kernel" in names) == (min(t for t in t_o if t) >= 9)
    cplx = lambda t: torch.view_as_complex(t.double().contiguous())  # noqa: E731
    got, go, w = cplx(x.grad.cpu()), cplx(go), cplx(w)
    offs = [0, 0, 0, 0]
    for l, (k, n) in enumerate(zip(t_ff, t_o)):
        m = 2 * l + 1
        h = go[:, offs[1]:offs[1] + n * m].reshape(bsz, n, m)
        v = w[offs[2]:offs[2] + k * n].reshape(n, k) / std[offs[3]:offs[3] + k]
        have = got[:, offs[0]:offs[0] + k * m].reshape(bsz, k, m)
        want = torch.einsum("ok,bom->bkm", v.conj(), h)
        # The division rounds a weight (2^-24), two pieces each factor (2^-23 of it, or 2^-39 of the largest of its row or
        # column), and 2 n products are added in fp32: at most 2^-24 of the sum of their moduli an addition, whatever the order.
        terms = torch.einsum("ok,bom->bkm", v.abs(), h.abs())
        least = 2. ** -38 * 2 * n * (v.abs().amax(0)[None, :, None] * h.abs().amax(1)[:, None, :] if n else 0.)
        assert ((have - want).abs() <= (2 ** -24 * (1 + 2 * n) + 2 ** -22) * 2 * terms + least).all(), l
        offs = [a + b for a, b in zip(offs, (k * m, n * m, k * n, k))]


@pytest.mark.parametrize("lmax,tin,tout,bsz,sparse", [
    (2, [3, 1, 2], [9, 9, 9], 1, False),
    (6, [16, 5, 9, 0, 2, 8, 12], [16, 12, 0, 13, 9, 10, 16], 5, False),
    (9, [4] * 10, [12] * 10, 3, True),
    (13, [9] * 14, [16] * 14, 2, False),
    (18, [2] * 19, [9] * 19, 1, False),
])
def test_layer_makes_the_same_gradient(dev, lmax, tin, tout, bsz, sparse):  # noqa: F811
    """Inside the layer and in the mixing's kernel the products are the same and are added in the same order."""
    from cgnet_amd import CG_layers
    torch.manual_seed(lmax)
    mod = CG_layers.CGBN_cuda(lmax, tin, tout, sparse_flag=sparse, device=dev)
    mod.eval()
    go = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(tout)), 2, generator=torch.Generator().manual_seed(1)).to(dev)
    grads = []
    for one_kernel in (False, True):
        mod.fused_backward = one_kernel
        x = rand_straight(tin, bsz, seed=lmax).float().to(dev).requires_grad_(True)
        out = mod(x, straight_output=True)
        names = _kernels(lambda: out.backward(go))
        assert "cg_backward_pair_kernel" in names and ("wmm_gradff_mfma_kernel" in names) != one_kernel
        grads.append(x.grad)
    assert torch.isfinite(grads[0]).all() and torch.equal(grads[0], grads[1])
