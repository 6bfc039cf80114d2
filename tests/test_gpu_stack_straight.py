"""A stack hands the straight tensor from layer to layer unless somebody looks at a layer's fragments: the numbers are the same, and
what a hook or a replaced forward sees is what it saw: lists of fragments."""
import pytest
import torch

from tests.test_gpu_parity import dev  # noqa: F401

pytestmark = pytest.mark.gpu


def _pass(net, x):
    for layer in net.cgs:
        layer.bnWMM.bn_cnt = 1.
    x = x.clone().requires_grad_(True)
    net.zero_grad(set_to_none=True)
    out = net(x)
    out.square().sum().backward()
    return [out.detach(), x.grad] + [p.grad for p in net.parameters() if p.requires_grad]


@pytest.mark.parametrize("skipconn", [True, False])
@pytest.mark.parametrize("bsz", [1, 3])
def test_straight_or_fragments(dev, monkeypatch, skipconn, bsz):  # noqa: F811
    from cgnet_amd import CG_layers, CGNet
    lmax, taus = 3, [[1] * 4, [4, 2, 3, 1], [2, 1, 1, 2], [3, 3, 1, 1]]
    torch.manual_seed(3)
    net = CGNet.SphericalCNN(lmax, taus, skipconn=skipconn).eval()
    x = torch.randn(bsz, 16, 2, device=dev)
    assert all(CG_layers.plain_call(layer) for layer in net.cgs)
    want = _pass(net, x)
    seen = []
    look = lambda module, args, out: seen.append([tuple(v.shape) for v in out])  # noqa: E731
    fragments = [[(bsz, t, 2 * l + 1, 2) for l, t in enumerate(ts)] for ts in taus[1:]]

    hook = net.cgs[1].register_forward_hook(look)
    got = _pass(net, x)
    hook.remove()
    assert seen == [fragments[1]] and all(torch.equal(a, b) for a, b in zip(got, want))

    seen.clear()
    hook = torch.nn.modules.module.register_module_forward_hook(
        lambda module, args, out: look(module, args, out) if isinstance(module, CG_layers.CGBN_cuda) else None)
    try:
        got = _pass(net, x)
    finally:
        hook.remove()
    assert seen == fragments and all(torch.equal(a, b) for a, b in zip(got, want))

    seen.clear()
    plain = CG_layers.CGBN_cuda.forward

    def wrapped(self, fs, straight_output=False):
        out = plain(self, fs, straight_output)
        look(self, None, out)
        return out
    with monkeypatch.context() as m:
        m.setattr(CG_layers.CGBN_cuda, "forward", wrapped)
        got = _pass(net, x)
    assert seen == fragments and all(torch.equal(a, b) for a, b in zip(got, want))
    assert all(CG_layers.plain_call(layer) for layer in net.cgs)


@pytest.mark.parametrize("skipconn", [True, False])
def test_arguments_of_the_next_layer(dev, skipconn):  # noqa: F811
    """What a layer's pre-hook, a module of another class in its place, or a hook on its product module takes in is a list of
    fragments, as the layer before it returns one."""
    from cgnet_amd import CG_layers, CGNet
    lmax, taus = 3, [[1] * 4, [4, 2, 3, 1], [2, 1, 1, 2], [3, 3, 1, 1]]
    torch.manual_seed(4)
    net = CGNet.SphericalCNN(lmax, taus, skipconn=skipconn).eval()
    x = torch.randn(2, 16, 2, device=dev)
    want = _pass(net, x)
    shapes = lambda fs: [tuple(v.shape) for v in fs]  # noqa: E731
    entering = [[(2, t, 2 * l + 1, 2) for l, t in enumerate(ts)] for ts in taus]
    seen = []

    hook = net.cgs[2].register_forward_pre_hook(lambda module, args: seen.append(shapes(args[0])))
    got = _pass(net, x)
    hook.remove()
    assert seen == [entering[2]] and all(torch.equal(a, b) for a, b in zip(got, want))

    class Other(torch.nn.Module):
        def __init__(self, layer):
            super().__init__()
            self.layer, self.bnWMM = layer, layer.bnWMM

        def forward(self, fs, straight_output=False):
            seen.append(shapes(fs))
            return self.layer(fs, straight_output)
    seen.clear()
    kept = net.cgs[1]
    net.cgs[1] = Other(kept)
    got = _pass(net, x)
    net.cgs[1] = kept
    assert seen == [entering[1]] and all(torch.equal(a, b) for a, b in zip(got, want))

    # the product module of a layer that chains product and mixing
    net.cgs[2].fused = False
    want = _pass(net, x)
    seen.clear()
    hook = net.cgs[2].cg.register_forward_hook(lambda module, args, out: seen.append(shapes(args[0])))
    got = _pass(net, x)
    hook.remove()
    assert seen == [entering[2]] and all(torch.equal(a, b) for a, b in zip(got, want))


def test_layer_with_other_outputs(dev):  # noqa: F811
    """A last layer with another number of output channels in its place: its degree 0 is taken as it is."""
    from cgnet_amd import CG_layers, CGNet
    lmax, taus = 2, [[1] * 3, [2, 2, 1], [2, 1, 1]]
    torch.manual_seed(5)
    net = CGNet.SphericalCNN(lmax, taus, skipconn=False)
    net.cgs[1] = CG_layers.CGBN_cuda(lmax, taus[1], [5, 1, 1], device=dev)
    net.eval()
    with torch.no_grad():
        x = torch.randn(3, 9, 2, device=dev)
        want = net.cgs[1](net.cgs[0](x))[0].reshape(3, -1)
        assert want.shape == (3, 10) and torch.equal(net(x), want)
