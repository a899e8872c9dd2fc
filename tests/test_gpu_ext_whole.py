"""The extended mode's whole-path kernel against the kernels per stage and bounce
(traversal = 1), bit for bit with equal counters: the two are the same device
functions in the same order per path. Image edges around a wave, one sample (finished
in the kernel) and several, waves smaller than the image, path lengths 0 and 1, scenes
with and without spheres, planes, sky and sphere lights, the features sink, served
waves, and which of the two forms runs: by scene, by size, by the memory there is."""
import json

import numpy as np
import pytest

import pathtracer_amd as pt
from pathtracer_amd import scenes


def plane_and_sky(spheres=3, light=True):
    """Spheres of the three materials over a ground plane under a sky, one of them a light."""
    s = scenes.random_spheres_dict(n=spheres, scene_seed=4, wavelengths=4, seed=9)
    s["quad"] = []
    s["plane"] = [{"position": [0.0, -0.2, 0.0], "materialID": 1, "lightID": 0}]
    s["environment"] = {"radiance": 0.7}
    if light:
        s["sphere"].append({"position": [0.5, 1.6, 0.3], "radius": 0.2, "materialID": 6, "lightID": 1})
    else:
        s["light"] = []
    return json.dumps(s)


def lens_scene():
    """The spheres' box with a lens in it, which the whole-path kernel does not take."""
    s = scenes.cornell_dict(4, seed=7)
    s["lens"] = [{"position": [0.5, 0.5, 0.4], "rotation": [0.0, 0.0, 0.0], "radius": 0.2, "focalLength": 0.3,
                  "thickness": 0.0, "isConverging": True, "materialID": 1, "lightID": 0}]
    return json.dumps(s)


SCENES = {
    "spheres": lambda: scenes.random_spheres(n=500, scene_seed=2, wavelengths=4, seed=7),
    "cornell1": lambda: scenes.cornell(1, seed=7),
    "plane_sky": plane_and_sky,
    "no_light": lambda: plane_and_sky(light=False),
    "quads_only": lambda: json.dumps(dict(scenes.cornell_dict(4, seed=7), sphere=[])),
    "sdf": lambda: scenes.sdf_scene(seed=3),
    "lens": lens_scene,
    "sdf_spheres": lambda: json.dumps(dict(json.loads(plane_and_sky()), sdf=json.loads(scenes.sdf_scene(seed=3))["sdf"])),
}
COUNTERS = ("sdf_steps", "sdf_exhausted", "segments", "shadow_segments", "paths", "nan_samples", "dispatches", "escaped", "emitter_hits", "lambert_hits",
            "dielectric_hits", "conductor_hits", "bvh_nodes", "shadow_bvh_nodes", "bad_refs")


def render(traversal, text, w, h, spp, depth, frames=2, wave_paths=0):
    with pt.Context(0, traversal=traversal, wave_paths=wave_paths) as ctx:
        r = pt.Renderer(ctx, ctx.scene_from_json(text), w, h, spf=spp, path_length=depth, mode=pt.MODE_EXT)
        for _ in range(frames):
            r.render_frame()
        ctx.profile(True)
        r.render_frame()
        names = set(ctx.profile_read())
        return r.acc.read(), ctx.counters(), names


def check(text, w, h, spp, depth, **k):
    a, ca, na = render(0, text, w, h, spp, depth, **k)
    b, cb, nb = render(1, text, w, h, spp, depth, **k)
    assert "k_ext_path" in na and "k_ext_path" not in nb
    np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
    assert {c: ca[c] for c in COUNTERS} == {c: cb[c] for c in COUNTERS}


@pytest.mark.gpu
@pytest.mark.parametrize("name", [n for n in SCENES if n != "lens"])
@pytest.mark.parametrize("spp", [1, 3])
def test_scenes(name, spp):
    check(SCENES[name](), 61, 37, spp, 7)


@pytest.mark.gpu
@pytest.mark.parametrize("w,h", [(1, 1), (63, 1), (65, 1)])
@pytest.mark.parametrize("spp", [1, 2])
def test_image_edges(w, h, spp):
    check(SCENES["spheres"](), w, h, spp, 5)


@pytest.mark.gpu
@pytest.mark.parametrize("depth", [0, 1])
def test_short_paths(depth):
    check(SCENES["plane_sky"](), 40, 30, 2, depth)


@pytest.mark.gpu
@pytest.mark.parametrize("spp", [1, 4])
def test_waves_smaller_than_the_image(spp):
    check(SCENES["spheres"](), 53, 41, spp, 4, wave_paths=1024)


@pytest.mark.gpu
@pytest.mark.parametrize("full_first", [False, True])
def test_features_and_a_full_wave_in_between(full_first):
    """First-hit features of both forms; and a context whose full wave (a scene the whole-path
    kernel does not take) serves the whole-path kernel afterwards, in place of a lean one or
    before there is one, with the cursors that wave holds, in dispatches and served waves."""
    text = SCENES["spheres"]()
    out = []
    for tr in (0, 1):
        with pt.Context(0, traversal=tr, graph_mode=1, wave_paths=8192) as ctx:  # what the full wave holds
            ctx.profile(True)
            ran = lambda: "k_ext_path" in ctx.profile_read(True)  # noqa: E731
            sc = ctx.scene_from_json(text)
            pc = pt.push_constants(45, 31, 3, 5)
            sc.camera(1, pc)
            pc.frame = pc.currentSamples = 3
            images = []
            for full in ((True, False, False) if full_first else (False, True, False)):
                if full:
                    lens = ctx.scene_from_json(lens_scene())
                    pt.Renderer(ctx, lens, 64, 48, spf=4, path_length=3, mode=pt.MODE_EXT).render_frame()
                    assert not ran()
                images.append(ctx.features(sc, pc))
                assert ran() == (tr == 0)
                with pt.Server(ctx) as server:
                    rid = server.submit(text, 24, 16, 8, 4, target=1e-6)
                    while server.step() is not None:
                        pass
                    images.append(np.asarray(server.read(rid)))
                assert ran() == (tr == 0)
            for x in images:
                np.testing.assert_array_equal(x.view(np.uint32), images[x.shape[-1] != pt.FEATURES].view(np.uint32))
            out.append(images[:2])
    for x, y in zip(*out):
        np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32))


def serve(traversal, names, **cfg):
    """Images, counters and kernel names (only of graph_mode 1: a graph's launches have none)."""
    with pt.Context(0, traversal=traversal, **cfg) as ctx, pt.Server(ctx) as server:
        ctx.profile(cfg.get("graph_mode") == 1)
        ids = [server.submit(SCENES[n](), 37 + 8 * k, 29, 6, 4 + k, target=1e-6) for k, n in enumerate(names)]
        while server.step() is not None:
            pass
        return [np.asarray(server.read(i)) for i in ids], ctx.counters(), set(ctx.profile_read())


def served_kernels(text, w, h, spp, min_spp=8, **cfg):
    """Images and kernel names of a served request (no graphs: their launches have no names)."""
    with pt.Context(0, graph_mode=1, **cfg) as ctx, pt.Server(ctx, min_spp=min_spp) as server:
        ctx.profile(True)
        rid = server.submit(text, w, h, spp, 4, target=1e-6)
        while server.step() is not None:
            pass
        return server.read(rid), set(ctx.profile_read())


@pytest.mark.gpu
@pytest.mark.parametrize("names", [["spheres", "plane_sky"], ["sdf", "spheres", "sdf_spheres", "quads_only", "sdf"]])
def test_batched_waves(names):
    """Requests of several scenes in one wave, with and without SDFs: the same images, from a
    captured graph and from launches one by one."""
    a, ca, _ = serve(0, names)
    g, cg, ng = serve(0, names, graph_mode=1)
    b, cb, nb = serve(1, names, graph_mode=1)
    assert "k_ext_path" in ng and "k_ext_path" not in nb
    for x, y, z in zip(a, g, b):
        np.testing.assert_array_equal(x.view(np.uint32), z.view(np.uint32))
        np.testing.assert_array_equal(y.view(np.uint32), z.view(np.uint32))
    assert {c: ca[c] for c in COUNTERS} == {c: cg[c] for c in COUNTERS} == {c: cb[c] for c in COUNTERS}


@pytest.mark.gpu
def test_a_wave_with_a_scene_the_kernel_does_not_take():
    """One lens among the requests: the wave runs the kernels per stage, with the same images as
    every form, and as the other requests get without it."""
    names = ["spheres", "sdf", "lens", "quads_only"]
    a, ca, na = serve(0, names, graph_mode=1)
    b, cb, _ = serve(1, names)
    alone, _, nl = serve(0, names[:2], graph_mode=1)
    assert "k_ext_path" not in na and "k_ext_path" in nl
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32))
    for x, y in zip(a, alone):
        np.testing.assert_array_equal(x.view(np.uint32), y.view(np.uint32))
    assert {c: ca[c] for c in COUNTERS} == {c: cb[c] for c in COUNTERS}


@pytest.mark.gpu
def test_no_room_for_the_batch_cursors():
    """The smallest budgets that serve a request beside a full wave have no room for the whole-path
    kernel's batch cursors: the kernels per stage serve it; with more room the kernel does."""
    text = SCENES["spheres"]()
    want, _ = served_kernels(text, 40, 24, 8, traversal=1)
    served = []
    paths, step = 1 << 16, 64 << 10
    for budget in range(FULL_PATH * paths, FULL_PATH * paths + (4 << 20), step):
        with pt.Context(0, graph_mode=1, wave_paths=paths, hbm_budget=budget) as ctx:
            try:
                lens = ctx.scene_from_json(lens_scene())
                pt.Renderer(ctx, lens, 64, 64, spf=16, path_length=2, mode=pt.MODE_EXT).render_frame()
                ctx.profile(True)
                with pt.Server(ctx) as server:
                    rid = server.submit(text, 40, 24, 8, 4, target=1e-6)
                    while server.step() is not None:
                        pass
                    got = np.asarray(server.read(rid))
            except pt.PTError as e:
                assert e.status == pt.PT_ERR_BUDGET and not served
                continue
            np.testing.assert_array_equal(got.view(np.uint32), np.asarray(want).view(np.uint32))
            served.append("k_ext_path" in ctx.profile_read())
        if served[-1]:
            break
    assert len(served) > 1 and served == [False] * (len(served) - 1) + [True]


FULL_PATH, LEAN_PATH = 336, 60  # bytes a path of the two waves


@pytest.mark.gpu
@pytest.mark.parametrize("ratio", [1.1, 4.0])
def test_budget_of_one_wave_serves_both_kinds_in_turn(ratio):
    """A dispatch of kernels per stage leaves its wave; a larger whole-path dispatch runs under a
    budget that holds the wave it would take alone (the full one, or the lean one) but not both."""
    w, h, spp = 512, 256, 4
    h2 = int(h * ratio)
    text = SCENES["spheres"]()
    want = render(0, text, w, h2, spp, 4, frames=0)[0]
    full, lean = FULL_PATH * w * h * spp, LEAN_PATH * w * h2 * spp
    one = FULL_PATH * w * h2 * spp if ratio < 2 else max(full, lean)
    rest = (w * h + w * h2) * 16 + (4 << 20)  # accumulators; scenes, cursors and counters
    assert one + (4 << 20) < full + lean
    with pt.Context(0, hbm_budget=one + rest) as ctx:
        lens = pt.Renderer(ctx, ctx.scene_from_json(lens_scene()), w, h, spf=spp, path_length=4, mode=pt.MODE_EXT)
        whole = pt.Renderer(ctx, ctx.scene_from_json(text), w, h2, spf=spp, path_length=4, mode=pt.MODE_EXT)
        ctx.profile(True)
        lens.render_frame()
        assert "k_ext_path" not in ctx.profile_read(True)
        first = lens.acc.read()
        for _ in range(2):
            whole.acc.reset()
            whole.frame = whole.current = 0
            whole.render_frame()
            assert "k_ext_path" in ctx.profile_read(True)
            np.testing.assert_array_equal(whole.acc.read().view(np.uint32), want.view(np.uint32))
            lens.acc.reset()
            lens.frame = lens.current = 0
            lens.render_frame()
            np.testing.assert_array_equal(lens.acc.read().view(np.uint32), first.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["spheres", "sdf"])
def test_a_small_wave_in_a_large_capacity(name):
    """What a served wave holds decides which kernels trace it, not what it could hold."""
    a, na = served_kernels(SCENES[name](), 64, 48, 8, wave_paths=1 << 26)
    b, nb = served_kernels(SCENES[name](), 64, 48, 8, traversal=1)
    assert "k_ext_path" in na and "k_ext_path" not in nb
    np.testing.assert_array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))


@pytest.mark.gpu
def test_large_sdf_waves_keep_the_kernels_per_stage():
    """Above 2^25 paths, a dispatch and a served wave (1920 x 1080, 17 samples: 35 M paths)."""
    text = SCENES["sdf"]()
    _, names = served_kernels(text, 1920, 1080, 17, min_spp=17, wave_paths=1 << 26)
    assert "k_ext_path" not in names and "k_ext_march_mandelbulb" in names
    assert "k_ext_path" not in render(0, text, 1920, 1080, 17, 2, frames=0)[2]
    assert "k_ext_path" in render(0, text, 1920, 1080, 16, 2, frames=0)[2]


@pytest.mark.gpu
@pytest.mark.parametrize("kinds,size,whole", [
    (("mandelbulb", "menger"), (1920, 1080, 8), True),  # 16.6 M paths
    (("mandelbulb", "menger"), (1920, 1080, 9), False),
    (("terrain", "mandelbulb"), (1920, 1080, 2), True),
    (("terrain",), (1280, 720, 4), True),  # 3.7 M
    (("terrain",), (1280, 720, 5), False),
    (("terrain", "blob"), (1280, 720, 5), False),
    (("blob",), (1920, 1080, 16), True),  # 33.2 M
    (("blob",), (1920, 1080, 17), False),
])
def test_sdfs_among_spheres_go_whole_up_to_a_size(kinds, size, whole):
    """Where the line lies, and the same images on both sides of it."""
    s = json.loads(SCENES["sdf_spheres"]())
    base = {d["kind"]: d for d in s["sdf"]}
    base["terrain"] = {"kind": "terrain", "position": [0, 0.5, 2.5], "boundingSize": [8, 6, 8], "material": 1.0}
    base["blob"] = dict(base["terrain"], kind="blob", position=[0, 1, 2.5], boundingSize=[3, 3, 3])
    s["sdf"] = [base[k] for k in kinds]
    w, h, spp = size
    a, _, na = render(0, json.dumps(s), w, h, spp, 3, frames=0)
    b, _, nb = render(1, json.dumps(s), w, h, spp, 3, frames=0)
    assert ("k_ext_path" in na) == whole and "k_ext_path" not in nb
    np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("graph_mode", [0, 1])
def test_a_served_wave_grows_a_full_one(graph_mode):
    """A full wave nearly as large as the served waves' capacity grows for them, which takes the
    batch cursors back: they are made after it. Before, between and after dispatches of both kinds."""
    text = SCENES["spheres"]()
    with pt.Context(0, wave_paths=16384, graph_mode=graph_mode) as ctx:
        lens, sc = ctx.scene_from_json(lens_scene()), ctx.scene_from_json(text)
        images = []
        for (w, h) in ((None, None), (120, 120), (128, 128), (16, 16)):
            if w:
                pt.Renderer(ctx, lens, w, h, spf=1, path_length=3, mode=pt.MODE_EXT).render_frame()
                pt.Renderer(ctx, sc, w, h, spf=1, path_length=3, mode=pt.MODE_EXT).render_frame()
            ctx.profile(graph_mode == 1)
            ctx.profile_read(True)
            with pt.Server(ctx) as server:
                rid = server.submit(text, 40, 24, 8, 4, target=1e-6)
                while server.step() is not None:
                    pass
                images.append(np.asarray(server.read(rid)))
            assert graph_mode == 0 or "k_ext_path" in ctx.profile_read(True)
            ctx.profile(False)
        for x in images[1:]:
            np.testing.assert_array_equal(x.view(np.uint32), images[0].view(np.uint32))
