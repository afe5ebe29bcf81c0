"""Rays that lie in a face plane of a node's box: a zero direction component whose origin is
on the plane. The slab test's product is 0 * inf there, and the ray is outside the box
unless the box is flat along that axis, whichever sign the zero has."""
import itertools

import numpy as np
import pytest

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu


def _scene(gpu, axis):
    """One triangle (u, v, w) = (-1, 0, 0), (1, 0, 0), (0, 1, 0), with u along `axis` and v the
    next one: its box spans [-1, 1] x [0, 1] and is flat along w."""
    v = np.roll(np.float32([[-1, 0, 0], [1, 0, 0], [0, 1, 0]]), axis, axis=1)
    f = np.int32([[0, 1, 2]])
    d = scenes.SceneDesc(nder=1, width=8, height=8, cam_to_world=scenes.look_at((0, 0.4, 3), (0, 0.4, 0), (0, 1, 0)),
                         cam_to_ndc=scenes.cam_to_ndc(45.0), shapes=[scenes.ShapeDesc(v, f, bsdf_id=0, light_id=0)],
                         bsdfs=[("diffuse", (0.5, 0.5, 0.5))], lights=[("area", 0, (3.0, 2.0, 1.0), True)], spp=1, max_bounces=1)
    return scenes.instantiate(gpu, d)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_a_ray_in_a_face_plane_is_outside_the_box(gpu, axis):
    """Rays along w: through the triangle's inside they hit, along its edge in the plane
    v = 0 (inside the triangle by the closest-hit test's tolerance of 1e-6, but in the low
    face of its box) they miss, as they do beside it."""
    sc = _scene(gpu, axis)
    rays, want = [], []
    for zu, zv, sign in itertools.product((0.0, -0.0), (0.0, -0.0), (1.0, -1.0)):
        for v, hit in ((2.0 ** -10, True), (0.25, True), (0.0, False), (-2.0 ** -10, False)):
            o, d = np.float32([0.125, v, -2.0 * sign]), np.float32([zu, zv, sign])
            rays.append([*np.roll(o, axis), *np.roll(d, axis), 1e-3, 1e30])
            want.append(hit)
    face, t = gpu.trace(sc, np.array(rays, np.float32))
    assert ((face == 0) == np.array(want)).all()
    assert (t[np.array(want)] == 2.0).all()


@pytest.mark.parametrize("kind", [1, 2, 3])
@pytest.mark.parametrize("spp", [8192, 163840])
def test_images_of_rays_in_face_planes_do_not_depend_on_where_the_tree_is(gpu, kind, spp):
    """Two emitting quads that meet in the plane x = 0 of a camera in that plane, in single precision,
    through the middle pixel of 32,769: at 16,384.5 a float has 1 / 512 to the next, so one jittered ray
    in 512 lies in the plane and misses both, whether the tree is in LDS or in HBM, for few
    samples and for many (two waves per SIMD hold 131,072)."""
    lv, lf = scenes.quad((-1.0, 0, 0), 2.0, 2, 1)
    rv, rf = scenes.quad((1.0, 0, 0), 2.0, 2, 1)
    assert lv[:, 0].max() == 0 and rv[:, 0].min() == 0
    before = gpu.precision()
    gpu.set_precision(32)
    try:
        d = scenes.SceneDesc(nder=1, width=32769, height=32769, cam_to_world=scenes.look_at((0, 0.125, 6), (0, 0.125, 0), (0, 1, 0)),
                             cam_to_ndc=scenes.cam_to_ndc(20.0), crop=(16384, 16384, 1, 1), spp=spp, max_bounces=1,
                             shapes=[scenes.ShapeDesc(lv, lf, bsdf_id=0, light_id=0), scenes.ShapeDesc(rv, rf, bsdf_id=0, light_id=1)],
                             bsdfs=[("diffuse", (0.0, 0.0, 0.0))], lights=[("area", 0, (1.0, 1.0, 1.0), True), ("area", 1, (1.0, 1.0, 1.0), True)])
        sc = scenes.instantiate(gpu, d)
    finally:
        gpu.set_precision(before)
    lds = scenes.render_primal(gpu, d, seed=5, scene=sc, kind=kind)
    gpu.set_tree_in_hbm(sc, True)
    hbm = scenes.render_primal(gpu, d, seed=5, scene=sc, kind=kind)
    assert np.allclose(lds, hbm, rtol=1e-6)
    miss = spp * (1.0 - float(lds[0, 0, 0]))   # binomial of mean spp / 512: within 5 sigma of it
    assert abs(miss - spp / 512) <= 5 * (spp / 512) ** 0.5
