"""Rays, triangles and coordinates at the ends of the FP32 range: what the
plain operators answer, the traversal's cheaper arithmetic answers too.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import cpu_ref  # noqa: E402
from gartus_amd import api, scenes  # noqa: E402
from gartus_amd.scene_data import DIFFUSE_LIGHT, LAMBERTIAN, SPHERE, TRIANGLE, Material, SceneData  # noqa: E402


def _scene(kind, rows, material):
    s = SceneData()
    s.add(kind, rows, s.add_material(material))
    return s


GREY = Material(LAMBERTIAN, (0.5, 0.5, 0.5))
LIGHT = Material(DIFFUSE_LIGHT, (2.0, 3.0, 4.0))


def _agrees_with_oracle(data, o, d):
    got = api.RayScene(data).with_bvh().intersect(o, d)
    ref = cpu_ref.Scene(data).intersect(o, d, use_bvh=False)
    np.testing.assert_array_equal(got["prim"], ref["prim"])
    np.testing.assert_allclose(got["t"], ref["t"], rtol=1e-6)
    return got


def test_directions_whose_reciprocal_is_subnormal():
    """1/d of a component from 2^126 on is below the normal range, not zero."""
    tris = np.array([[-0.5, -0.5, z, 0.5, -0.5, z, 0.0, 0.5, z] for z in -3e36 * np.arange(1, 31)])
    data = _scene(TRIANGLE, tris.astype(np.float32).astype(np.float64), GREY)
    o = np.array([[0.0, -0.25, 0.0], [0.1, -0.4, -4e36], [0.0, -0.25, -8.5e37]], np.float32)
    d = np.array([[0.0, 0.0, -1e38], [0.0, 0.0, -2e38], [0.0, 0.0, 1.5e38]], np.float32)
    got = _agrees_with_oracle(data, o, d)
    assert (got["prim"] >= 0).all() and got["t"][0] == pytest.approx(0.03, rel=1e-5)


def _huge_triangle(material):
    return _scene(TRIANGLE, [[-3e12, -3e12, -1e12, 7e12, -3e12, -1e12, -3e12, 7e12, -1e12]], material)


def test_triangle_determinants_beyond_the_reciprocals_range():
    """|e1 . (d x e2)| of 1e38: a triangle of 1e13 met at t = 1 by a direction of 1e12."""
    data = _huge_triangle(GREY).as_float32_exact()
    o = np.zeros((3, 3), np.float32)
    d = np.array([[0.0, 0.0, -1e12], [1e11, 2e11, -1e12], [1.2e12, -1e12, -1.3e12]], np.float32)
    got = _agrees_with_oracle(data, o, d)
    assert (got["prim"] == 0).all() and got["t"][0] == pytest.approx(1.0, rel=1e-5)


def test_renders_of_huge_triangles():
    """The same triangle in a render, whose camera rays are as long as its focus distance."""
    scene = api.RayScene(_huge_triangle(LIGHT)).with_bvh()
    c = scenes.camera_record(dict(width=24, aspect=1.0, spp=2, depth=1, vfov=20.0, lookfrom=(0.0, 0.0, 0.0),
                                  lookat=(0.0, 0.0, -1.0)))
    c.focus_distance = 1e12
    camera = api.RayCamera.__new__(api.RayCamera)
    camera.raw = c
    px = api.PathTracer(camera).render_hdr_image(scene).pixels
    np.testing.assert_array_equal(px, np.broadcast_to(np.float32([2.0, 3.0, 4.0]), px.shape))


def test_renders_with_directions_whose_square_is_beyond_the_reciprocals_range():
    """|d|^2 of 1.3e38 against a sphere: powers of two keep every step of the test exact, and the hit (at its
    centre to FP32, so it emits nothing) is told from a miss by the background."""
    scale = 1.25 * 2.0 ** 63
    z = -1.25 * 2.0 ** 57
    scene = api.RayScene(_scene(SPHERE, [[0.0, 0.0, z, 1.0]], LIGHT)).with_bvh()
    d = np.array([[0.0, 0.0, -scale]], np.float32)
    assert scene.intersect(np.zeros((1, 3), np.float32), d)["prim"][0] == 0
    c = scenes.camera_record(dict(width=4, aspect=1.0, spp=1, depth=1, vfov=1e-18, lookfrom=(0.0, 0.0, 0.0),
                                  lookat=(0.0, 0.0, -1.0)))
    c.focus_distance = scale
    camera = api.RayCamera.__new__(api.RayCamera)
    camera.raw = c
    px = api.PathTracer(camera).render_hdr_image(scene).pixels
    np.testing.assert_array_equal(px, 0.0)


def test_the_sign_of_zero_survives_a_normal():
    """A sphere's u at the seam (outward = (-1, 0, -0)) is atan2 of a signed zero: 1, not 0."""
    data = _scene(SPHERE, [[0.0, 0.0, 0.0, 1.0]], GREY)
    o = np.array([[-5.0, 0.0, -0.0], [-5.0, 0.0, 0.0]], np.float32)
    d = np.array([[1.0, 0.0, -0.0], [1.0, 0.0, 0.0]], np.float32)
    got = _agrees_with_oracle(data, o, d)
    ref = cpu_ref.Scene(data).intersect(o, d)
    np.testing.assert_allclose(got["u"], ref["u"], rtol=0, atol=1e-6)
    np.testing.assert_array_equal(got["u"], np.float32([1.0, 0.0]))
