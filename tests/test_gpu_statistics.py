"""Running stds of the stand-alone fragment norm (fn_stats_kernel, fn_update_std_kernel) at the edges of its units: 64, 32 and
16 channels a wave by the length of a row, one channel over, several samples a stage, groups of samples of unequal size."""
import pytest
import torch

from tests.test_gpu_parity import dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax,t_ff,bsz", [
    (0, {0: 65}, 1),
    (0, {0: 7}, 200),                                      # rows of one entry: many samples a stage
    (3, {0: 64, 1: 1, 2: 129, 3: 5}, 9),                   # nine samples in eight groups
    (12, {11: 64, 12: 33}, 17),                            # rows of 23 (64 channels a wave) and 25 (32 a wave)
    (24, {23: 32, 24: 17}, 3),                             # rows of 47 and 49 (16 a wave)
    (47, {47: 16, 2: 300}, 2),
])
def test_running_stds(dev, lmax, t_ff, bsz):  # noqa: F811
    from cgnet_amd import CG_layers
    t_ff = [t_ff.get(l, 0) for l in range(lmax + 1)]
    mod = CG_layers.MyBatchNormWeightMM_cuda(lmax, t_ff, [1 if t else 0 for t in t_ff])
    g = torch.Generator().manual_seed(lmax + bsz)
    old = torch.rand(sum(t_ff), generator=g)
    ff = torch.randn(bsz, sum(t * (2 * l + 1) for l, t in enumerate(t_ff)), 2, generator=g) + 0.5
    with torch.no_grad():
        mod.bn_stds.copy_(old)
    mod.bn_cnt = 3.
    mod(ff.to(dev))
    o, want = 0, []
    for l, t in enumerate(t_ff):
        n = t * (2 * l + 1)
        z = ff[:, o:o + n].double().pow(2).sum(-1).sqrt().reshape(bsz, t, 2 * l + 1)
        want.append(z.var((0, 2), unbiased=False).sqrt())
        o += n
    want = 0.75 * old.double() + 0.25 * torch.cat(want)
    # |z| is rounded to float32 (half an ulp, 6e-8, in a spread of its own size), the result twice
    assert torch.allclose(mod.bn_stds.detach().cpu().double(), want, rtol=5e-7, atol=5e-7)
    assert mod.bn_cnt == 4.
