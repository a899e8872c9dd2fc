"""The persistent reference-mode kernel at the sizes where its queue and its two
ways out can go wrong, bit for bit against the CPU restatement: fewer paths than
lanes, one more or less than a wave, ragged images, one sample per pixel
(finished in the kernel) and several (the fold), waves smaller than the image,
path lengths 0 and 1, and scenes with SDF objects of each kind and of mixed kinds.
Also the kernel's integer powers against ptm_pow, on the CPU."""
import ctypes as C
import json
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

import pathtracer_amd as pt
from oracle import ptref

ROOT = Path(__file__).resolve().parent.parent
GOLDEN = ROOT / "tests" / "golden" / "scenes"


def sdf_scene(kinds):
    """scene0 with SDF objects of these kinds in front of its camera."""
    s = json.loads((GOLDEN / "scene0.json").read_text())
    extra = {"mandelbulb": {"iterations": 8, "bailout": 16.0}, "menger": {"iterations": 3}}
    s["sdf"] = [dict({"kind": k, "position": [2.0 + 1.5 * i, 1.3, 0.5 - i], "boundingSize": [2.2, 2.2, 2.2],
                      "material": 1.0}, **extra.get(k, {})) for i, k in enumerate(kinds)]
    return json.dumps(s)


def both(text, w, h, spf, depth, frames=1, wave_paths=0):
    """(GPU texels, counters), (oracle texels, counters) after `frames` dispatches."""
    with pt.Context(0, wave_paths=wave_paths) as ctx:
        sc = ctx.scene_from_json(text)
        r = pt.Renderer(ctx, sc, w, h, spf=spf, path_length=depth)
        for _ in range(frames):
            r.render_frame()
        got, gc = r.acc.read(), ctx.counters()
    pc = pt.push_constants(w, h, spf=spf, path_length=depth)
    ubo, pc, sdfs = pt.pack_json(text, 1, pc)
    blob = b"".join(bytes(s) for s in sdfs)
    ref = np.zeros((h, w, 4), np.float32)
    tot = {}
    for f in range(frames):
        pc.frame = pc.currentSamples = (f + 1) * spf
        for k, v in ptref.dispatch(bytes(ubo), bytes(pc), blob, len(sdfs), ref).items():
            tot[k] = tot.get(k, 0) + v
    return (got, gc), (ref, tot)


def check(*a, **k):
    (got, gc), (ref, rc) = both(*a, **k)
    np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))
    for key in ("segments", "shadow_segments", "sdf_steps"):
        assert gc[key] == rc[key], key
    return gc


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(1, 1), (63, 1), (64, 1), (65, 1), (37, 29)])
@pytest.mark.parametrize("spf", [1, 3])
def test_image_edges(w, h, spf):
    gc = check((GOLDEN / "scene0.json").read_text(), w, h, spf, 5, frames=2)
    assert gc["paths"] == w * h * spf * 2 and gc["dispatches"] == 2


@pytest.mark.gpu
@pytest.mark.parametrize("depth", [0, 1])
def test_short_paths(depth):
    check((GOLDEN / "scene2.json").read_text(), 40, 30, 2, depth)


@pytest.mark.gpu
@pytest.mark.parametrize("spf", [1, 5])
def test_waves_smaller_than_the_image(spf):
    """1024-path waves: pixel chunks of 1024 and samples in several waves each."""
    check(sdf_scene(["menger"]), 61, 43, spf, 4, wave_paths=1024)


@pytest.mark.gpu
@pytest.mark.parametrize("kinds", [["mandelbulb"], ["menger"], ["blob"], ["terrain"], ["blob", "menger", "mandelbulb"],
                                   ["menger", "menger"]], ids="-".join)
def test_sdf_kinds(kinds):
    check(sdf_scene(kinds), 96, 80, 2, 5)


@pytest.mark.gpu
def test_a_larger_dispatch_allocates_nothing():
    """After a context's first dispatch its wave is there: a larger one takes no device memory."""
    with pt.Context(0) as ctx:
        sc = ctx.scene_from_json((GOLDEN / "scene0.json").read_text())
        r = [pt.Renderer(ctx, sc, w, h, spf=2, path_length=3) for w, h in ((32, 24), (640, 480), (1920, 1080))]
        free, total = C.c_size_t(), C.c_size_t()
        left = []
        for x in r:
            x.render_frame()
            ctx.sync()
            assert pt.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
            left.append(free.value)
        assert left[1:] == left[:1] * 2


POW_C = r"""
#include "ptmath.h"
void slow(const float* x, float* o, int n, float e) { for (int i = 0; i < n; ++i) o[i] = ptm_pow(x[i], e); }
void m5(const float* x, float* o, int n) { for (int i = 0; i < n; ++i) o[i] = ptm_pow_m5(x[i]); }
/* the device code's r^7 of the middle range (mandelbulb_terms) */
int p7(const float* x, float* o, int n) {
    int slow = 0;
    for (int i = 0; i < n; ++i) {
        double d = (double)x[i], d2 = d * d, d3 = d2 * d, y = d3 * d3 * d;
        o[i] = (float)y;
        uint32_t dropped = (uint32_t)ptm_d2u(y) & 0x1fffffffu;
        if (dropped - (0x10000000u - 8192u) <= 2u * 8192u) { ++slow; o[i] = (float)ptm__exp_d(7.0 * ptm__log_d(d)); }
    }
    return slow;
}
"""


def test_integer_powers_equal_ptm_pow(tmp_path):
    """ptm_pow_m5 and the mandelbulb's r^7 give ptm_pow's binary32 value: over random
    values of their ranges, the ends, and for m5 zeros, infinities, NaN and denormals."""
    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("gcc not found")
    (tmp_path / "p.c").write_text(POW_C)
    so = tmp_path / "p.so"
    subprocess.run([gcc, "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", str(ROOT / "pathtracer_amd" / "csrc"),
                    str(tmp_path / "p.c"), "-o", str(so), "-lm"], check=True)
    lib = C.CDLL(str(so))
    fp = C.POINTER(C.c_float)
    rng = np.random.default_rng(5)
    ptr = lambda a: a.ctypes.data_as(fp)  # noqa: E731

    def slow(x, e):
        o = np.empty_like(x)
        lib.slow(ptr(x), ptr(o), x.size, C.c_float(e))
        return o

    x = np.exp2(rng.uniform(-16, 16, 1_500_000)).astype(np.float32)
    x = np.concatenate([x, np.float32([2.0 ** -16, 2.0 ** 16, 1.0, 1.0000001, 0.99999994, 3.0, 1.5])])
    o = np.empty_like(x)
    taken = lib.p7(ptr(x), ptr(o), x.size)
    np.testing.assert_array_equal(o.view(np.uint32), slow(x, 7.0).view(np.uint32))
    assert taken > 0, "the near-boundary path was not exercised"
    # wavelengths in metres, then the whole binary32 range and its special values
    l = (rng.uniform(360.0, 830.0, 500_000).astype(np.float32) * np.float32(1e-9)).astype(np.float32)
    a = rng.integers(0, 2 ** 32, 500_000, dtype=np.uint64).astype(np.uint32).view(np.float32)
    s = np.float32([0.0, -0.0, 1.0, -1.0, np.inf, -np.inf, np.nan, 1e-45, 1e-38, 3.4e38, 2.0, 0.5])
    for x in (l, a, s):
        o = np.empty_like(x)
        lib.m5(ptr(x), ptr(o), x.size)
        want = slow(x, -5.0)
        same = (o.view(np.uint32) == want.view(np.uint32)) | (np.isnan(o) & np.isnan(want))
        assert same.all(), x[~same][:5]
