"""Feature images finished on the device, and the context's scratch memory: the
means against the library's own sums of one-sample images, whatever the waves;
scratch given back when another allocation needs its room under the budget."""
import numpy as np
import pytest

import pathtracer_amd as pt
from pathtracer_amd import scenes


def features(w, h, spp, wave_paths=0):
    with pt.Context(0, wave_paths=wave_paths) as ctx:
        sc = ctx.scene_from_json(scenes.random_spheres(n=40, scene_seed=3, wavelengths=4, seed=3))
        pc = pt.push_constants(w, h, spp, 4)
        sc.camera(1, pc)
        one = []
        for k in range(spp):
            pc.samplesPerFrame, pc.frame, pc.currentSamples = 1, k + 1, 1
            one.append(ctx.features(sc, pc))
        pc.samplesPerFrame = pc.frame = pc.currentSamples = spp
        return ctx.features(sc, pc), one


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (64, 4, 2), (37, 29, 5)])
def test_means_of_one_sample_images(w, h, spp):
    """The n-sample image's channels are the means of its one-sample images: FP32 sums
    of n terms and one division, 4 n units of 2^-24 of the terms' size; the standard
    error of Y from the same samples in binary64 (its sums of Y and Y^2 are FP32, so
    relative to the mean's size)."""
    got, one = features(w, h, spp)
    stack = np.stack(one).astype(np.float64)
    tol = 4 * spp * 2.0 ** -24
    mean = stack[..., :10].mean(0)
    assert np.all(np.abs(got[..., :10] - mean) <= tol * np.abs(stack[..., :10]).mean(0) + 1e-30)
    assert np.all(got[..., 11] == spp)
    y = stack[..., 1]
    if spp > 1:
        se2 = y.var(0, ddof=1) / spp
        assert np.all(np.abs(got[..., 10].astype(np.float64) ** 2 - se2) <= 8 * tol * (y ** 2).sum(0) + 1e-30)
    else:
        assert np.all(got[..., 10] == 0)
    small, _ = features(w, h, spp, wave_paths=1024)
    np.testing.assert_array_equal(got.view(np.uint32), small.view(np.uint32))


@pytest.mark.gpu
def test_scratch_gives_way_under_the_budget():
    """A resolve keeps 3 bytes a pixel; an accumulator that fits the budget only
    without them is still made, and the resolve then refused as before."""
    w = h = 1024
    with pt.Context(0, hbm_budget=w * h * 16 + w * h * 4) as ctx:
        acc = ctx.accum(w, h)
        first = acc.resolve_srgb8()
        extra = ctx.accum(w // 2, h // 2)  # 4 MB: the whole rest
        with pytest.raises(pt.PTError) as e:
            acc.resolve_srgb8()
        assert e.value.status == pt.PT_ERR_BUDGET
        extra.release()
        np.testing.assert_array_equal(acc.resolve_srgb8(), first)
