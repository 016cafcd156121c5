"""A render walks its scene with one search (resumable, shared by a wave's rays), a query with another. They visit the
same nodes, test the same primitives and choose the same hits, with binary and with four-wide nodes, alone and in a
batch; and the counting, four-wide and batched forms of the render's kernels answer like the plain ones.
"""
import contextlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from gartus_amd import abi, api, scenes  # noqa: E402
from gartus_amd.scene_data import DIFFUSE_LIGHT, Material, SceneData  # noqa: E402


def _camera(spec, w, h):
    c = api.RayCamera.__new__(api.RayCamera)
    c.raw = scenes.camera_record(dict(spec, width=w, aspect=w / (h + 0.5)))
    if "nee" in spec:
        c.raw.direct_lighting_mode = abi.GT_LIGHTING_NEE
    return c


@contextlib.contextmanager
def _tuned(ctx, **kw):
    old = ctx.tuning
    ctx.set_tuning(**kw)
    try:
        yield
    finally:
        ctx.set_tuning(**{k: getattr(old, k) for k in kw})


def _lit(data):
    """The scene with every primitive a light of its own colour."""
    s = SceneData()
    for i, (kind, row, _) in enumerate(data.primitives()):
        s.add(kind, [row], s.add_material(Material(DIFFUSE_LIGHT, (1.0 + i % 61, 1.0 + i // 61 % 61, 1.0 + i // 3721))))
    return s.as_float32_exact()


SCENES = {
    "triangles": lambda: (scenes.terrain(grid=24, n_spheres=40)[0], (0.0, 14.0, 30.0), (0.0, 2.0, 0.0)),
    "mixed": lambda: (scenes.randomized_ray_scene(3), (0.0, 0.0, 4.0), (0.0, 0.0, -4.0)),
    "quads": lambda: (scenes.cornell()[0], (278.0, 278.0, -800.0), (278.0, 278.0, 0.0)),
    "spheres": lambda: (scenes.final_scene(), (13.0, 2.0, 3.0), (0.0, 0.0, 0.0)),
}


@pytest.mark.parametrize("width", [2, 4])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_a_renders_first_hits_are_the_queries(name, width):
    """The albedo image takes its camera rays' hits from the query's search, the beauty image from the render's: where
    every primitive is a light of its own colour and a path ends at its first hit, a front side shows the same
    colour in both."""
    data, eye, at = SCENES[name]()
    scene = api.RayScene(_lit(data)).with_bvh()
    cam = _camera(dict(spp=1, depth=1, vfov=50.0, lookfrom=eye, lookat=at, background=(0.25, 0.5, 0.75)), 193, 151)
    with _tuned(scene.context, bvh_width=width):
        aovs = api.PathTracer(cam)._render_aovs(scene, cam)
        beauty = api.PathTracer(cam)._render(scene, cam).pixels.reshape(-1, 3)
    albedo, beauty2 = aovs.albedo_linear.reshape(-1, 3), aovs.beauty_linear.reshape(-1, 3)
    np.testing.assert_array_equal(beauty, beauty2)
    hit = albedo[:, 0] > 0
    np.testing.assert_array_equal(beauty[~hit], np.broadcast_to(np.float32([0.25, 0.5, 0.75]), beauty[~hit].shape))
    front = hit & (beauty[:, 0] > 0)
    np.testing.assert_array_equal(beauty[front], albedo[front])
    np.testing.assert_array_equal(beauty[hit & ~front], 0.0)  # a back side emits nothing
    assert hit.sum() > 2000 and front.sum() > 0.4 * hit.sum() and len(np.unique(albedo[front], axis=0)) >= 8


def _pinholes(rng, n, lo, hi):
    """n cameras of one pixel so narrow that their ray is known, and the rays."""
    cams, o, d = [], [], []
    for _ in range(n):
        eye, at = rng.uniform(lo, hi), rng.uniform(lo, hi)
        cams.append(_camera(dict(spp=1, depth=1, vfov=1e-13, lookfrom=tuple(eye), lookat=tuple(at)), 1, 1))
        fwd = (at - eye) / np.linalg.norm(at - eye)
        o.append(eye.astype(np.float32))
        d.append((eye + fwd).astype(np.float32) - eye.astype(np.float32))  # focus distance 1
    return cams, np.array(o), np.array(d)


@pytest.mark.parametrize("width", [2, 4])
@pytest.mark.parametrize("batched", [False, True], ids=["single", "batched"])
def test_counted_work_is_the_queries(width, batched):
    """Nodes fetched and primitives tested by counting renders of one ray each, against the query's statistics."""
    data = scenes.terrain(grid=48, n_spheres=60, seed=4)[0]
    scene = api.RayScene(_lit(data)).with_bvh()
    cams, o, d = _pinholes(np.random.default_rng(8), 96, (-40, 1, -40), (40, 9, 40))
    with _tuned(scene.context, bvh_width=width, count_traversal=1):
        want = scene.intersect(o, d, with_stats=True)
        if batched:
            images, stats = api.render_batch([(scene, c, None, None) for c in cams], stats=True)
            images = [im.pixels for im in images]
        else:
            images, stats = [], dict.fromkeys(("ext_node_fetches", "ext_prim_tests", "extension_rays"), 0)
            for c in cams:
                im, st = api.PathTracer(c)._render(scene, c, stats=True)
                images.append(im.pixels)
                for k in stats:
                    stats[k] += st[k]
    hits = want["prim"] >= 0
    assert 10 < hits.sum() < len(cams)
    st = want["stats"]
    assert stats["extension_rays"] == len(cams)
    assert stats["ext_node_fetches"] * width + len(cams) == st["node_bounds_tests"]
    assert stats["ext_prim_tests"] == st["primitive_candidates"]
    seen = np.array([not np.array_equal(im.reshape(3), np.float32([0.7, 0.8, 1.0])) for im in images])
    np.testing.assert_array_equal(seen, hits)


def _connecting():
    """(scene, lights, environment, camera spec) of each kind of shadow ray, several scenes for a batch."""
    out = []
    for seed in (1003, 1004):
        data, lights, cam = scenes.batch_scene(seed)
        targets = api.SamplingTargetList()
        for _, q, _ in lights:
            targets.add_quad(q[0:3], q[3:6], q[6:9])
        out.append((api.RayScene(data).with_bvh(), targets, None, dict(cam, spp=3, nee=True)))
    for n in (12, 150):
        data, env, cam = scenes.ggx_environment(n_random=n, env_size=(64, 32))
        out.append((api.RayScene(data).with_bvh(), None, api.EnvironmentLight.from_rgb32f(env), dict(cam, spp=3, nee=True)))
    return out


@pytest.mark.parametrize("width", [2, 4])
def test_counting_and_batched_renders_are_the_plain_ones(width):
    """Every form of the extend and connect kernels with the same nodes gives the same image, bit for bit."""
    items = [(s, _camera(spec, 83, 47), lights, env) for s, lights, env, spec in _connecting()]
    ctx = items[0][0].context
    with _tuned(ctx, bvh_width=width):
        plain = [api.PathTracer(c)._render(s, c, lights, env).pixels for s, c, lights, env in items]
        batch = [im.pixels for im in api.render_batch(items)]
        with _tuned(ctx, count_traversal=1):
            counted, sums = [], dict.fromkeys(("ext_node_fetches", "ext_prim_tests", "shadow_node_fetches",
                                               "shadow_prim_tests", "shadow_rays"), 0)
            for s, c, lights, env in items:
                im, st = api.PathTracer(c)._render(s, c, lights, env, stats=True)
                counted.append(im.pixels)
                assert st["shadow_rays"] > 0 and st["shadow_prim_tests"] > 0
                for k in sums:
                    sums[k] += st[k]
            counted_batch, st = api.render_batch(items, stats=True)
    for k in range(len(items)):
        assert np.isfinite(plain[k]).all() and plain[k].std() > 0
        for other in (batch[k], counted[k], counted_batch[k].pixels):
            np.testing.assert_array_equal(other, plain[k], err_msg=f"scene {k}")
    assert {k: st[k] for k in sums} == sums


def test_four_wide_connections_render_the_binary_trees_images():
    """Node width changes the order of visits only. Only rays that meet two primitives at one distance may tell."""
    for s, lights, env, spec in _connecting():
        cam = _camera(spec, 83, 47)
        images = []
        for width in (2, 4):
            with _tuned(s.context, bvh_width=width):
                images.append(api.PathTracer(cam)._render(s, cam, lights, env).pixels.reshape(-1, 3))
        assert (images[0] == images[1]).all(axis=1).mean() > 0.995
