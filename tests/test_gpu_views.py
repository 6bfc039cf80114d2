"""The fragments one layer hands to the next are taken as the straight tensor they are views of, whatever dimensions have size
one; anything else is concatenated.  Evaluation without gradients gives what evaluation with them gives."""
import pytest
import torch

from tests.test_gpu_parity import dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bsz", [1, 3])
@pytest.mark.parametrize("taus", [[1], [2, 1, 3], [1, 1], [2, 0, 1]])
def test_straight_of_views(dev, bsz, taus):  # noqa: F811
    from cgnet_amd import CGutils
    from cgnet_amd.CG_layers import _straight
    x = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(taus)), 2, device=dev)
    parts = CGutils.reshape_out(x, taus)
    assert _straight(parts) is x
    for l, t in enumerate(taus):
        if t:
            # same sizes, not this place: another tensor, m reversed in memory, samples swapped
            for other in (parts[l].clone(), parts[l].flip(2), parts[l].flip(0)):
                got = _straight(parts[:l] + [other] + parts[l + 1:])
                assert got is not x
                assert torch.equal(got, torch.cat([v.reshape(bsz, -1, 2) for v in parts[:l] + [other] + parts[l + 1:]], dim=1))
    half = CGutils.reshape_out(x[:, :taus[0]], taus[:1])          # the views stop short of the tensor's end
    assert torch.equal(_straight(half), x[:, :taus[0]])


def test_straight_of_transposed_views(dev):  # noqa: F811
    from cgnet_amd.CG_layers import _straight
    x = torch.randn(2, 9, 2, device=dev)
    swapped = x.view(2, 3, 3, 2).transpose(1, 2)                   # three channels of degree 1, m and channel exchanged
    assert torch.equal(_straight([swapped]), swapped.reshape(2, 9, 2))


@pytest.mark.parametrize("taus,bsz", [([2, 1, 2], 1), ([12] * 6, 3)])
def test_evaluation_without_gradients(dev, taus, bsz):  # noqa: F811
    from cgnet_amd import CG_layers
    net = CG_layers.CGBN_cuda(len(taus) - 1, taus, taus).eval()
    net.fused_inference = False
    x = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(taus)), 2, device=dev)
    want = net(x, straight_output=True)
    want.square().sum().backward()
    assert net.bnWMM.W.grad.abs().sum() > 0
    stds = net.bnWMM.bn_stds.clone()
    with torch.no_grad():
        assert torch.equal(net(x, straight_output=True), want)
    assert torch.equal(net.bnWMM.bn_stds, stds)
