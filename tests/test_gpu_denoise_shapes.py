"""The denoiser's weight-gradient and convolution kernels at ragged sizes: images
smaller than a tile, one more than a tile, several images; gradients against the
FP64 oracle, bit-equal from run to run, the atomics they fall back to without memory
for partial sums, and images computed alone (small tiles) and in a batch (large ones)."""
import numpy as np
import pytest

import pathtracer_amd as pt
from oracle import denoise_ref as D
from tests.test_denoise import random_features, random_params

SHAPES = [(1, 4, 4), (2, 12, 36), (3, 20, 68), (1, 64, 100)]


def setup(n, h, w, seed=11):
    rng = np.random.default_rng(seed)
    return (random_params(rng).astype(np.float32), random_features(rng, n, h, w),
            np.exp(rng.normal(-1.0, 1.0, (n, h, w, 3))).astype(np.float32))


def gradients(ctx, n, h, w, p, feat, target):
    with pt.Denoiser(ctx, n, h, w) as dn:
        dn.set_params(p)
        dn.set_loss(pt.DN_LOSS_L2)
        return dn.gradients(feat, target)


@pytest.mark.gpu
@pytest.mark.parametrize("n,h,w", SHAPES)
def test_gradients_at_ragged_sizes(gpu_ctx, n, h, w):
    """BF16 operands (relative error 2^-9 each) through 22 layers, forward and back:
    about 2 % of a gradient's norm, a cosine of 0.9998; the bar is the network's own, 0.995."""
    p, feat, target = setup(n, h, w)
    loss, g = gradients(gpu_ctx, n, h, w, p, feat, target)
    loss2, g2 = gradients(gpu_ctx, n, h, w, p, feat, target)
    np.testing.assert_array_equal(g.view(np.uint32), g2.view(np.uint32))
    ref_loss, ref = D.loss_and_grad(p.astype(np.float64), feat.astype(np.float64), target.astype(np.float64), "l2")
    assert abs(loss - ref_loss) <= 0.01 * ref_loss
    assert float(g.astype(np.float64) @ ref / (np.linalg.norm(g) * np.linalg.norm(ref))) > 0.995


@pytest.mark.gpu
def test_atomics_without_memory_for_partials():
    """A budget that holds the denoiser but not the partial sums: the same gradients but
    for the order of FP32 sums over 20 x 68 x 3 pixels (2^-24 each, at most 4080 terms)."""
    n, h, w = 3, 20, 68
    p, feat, target = setup(n, h, w)
    with pt.Context(0) as ctx:
        ctx.profile(True)
        _, g = gradients(ctx, n, h, w, p, feat, target)
        assert "k_dn_grad_sum" in ctx.profile_read()
    with pt.Context(0, hbm_budget=20 << 20) as ctx:  # the denoiser takes 17 MB, the partials more than the rest
        ctx.profile(True)
        _, a = gradients(ctx, n, h, w, p, feat, target)
        assert "k_dn_grad_sum" not in ctx.profile_read()
    assert np.linalg.norm(a - g) <= 4080 * 2.0 ** -24 * np.linalg.norm(g)


@pytest.mark.gpu
def test_a_batch_equals_its_images(gpu_ctx):
    rng = np.random.default_rng(5)
    feat = random_features(rng, 24, 96, 160)
    with pt.Denoiser(gpu_ctx, 24, 96, 160) as dn:
        dn.set_params(random_params(rng).astype(np.float32))
        batch = dn.denoise(feat)
        for i in (0, 7, 23):
            np.testing.assert_array_equal(dn.denoise(feat[i:i + 1])[0].view(np.uint32), batch[i].view(np.uint32))
