"""Closest-hit traversal where its per-ray setup and its stack can go wrong: rays along the
axes with zero components of either sign, and the smallest trees."""
import itertools

import numpy as np
import pytest

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu


def _closest(v, f, rays):
    """Brute force in float64: distance to the nearest triangle (inf: none) of each ray."""
    best = np.full(len(rays), np.inf)
    o, d, lo, hi = rays[:, :3].astype(np.float64), rays[:, 3:6].astype(np.float64), rays[:, 6], rays[:, 7]
    for a, b, c in f:
        e1, e2 = (v[b] - v[a]).astype(np.float64), (v[c] - v[a]).astype(np.float64)
        p = np.cross(d, e2)
        det = p @ e1
        with np.errstate(divide="ignore", invalid="ignore"):   # parallel rays: no hit
            s = o - v[a]
            u = (s * p).sum(1) / det
            q = np.cross(s, e1)
            w = (d * q).sum(1) / det
            t = (q @ e2) / det
            ok = (det != 0) & (u >= 0) & (w >= 0) & (u + w <= 1) & (t >= lo) & (t <= hi)
        best = np.where(ok & (t < best), t, best)
    return best


def test_axis_rays_with_zero_components_of_either_sign(gpu):
    """Origins off every box plane and off every edge, directions with two zero components
    (+0 and -0), in front of, beside and behind each shape: the hit and its distance are
    those of a brute-force test (distances are sums of fp32 products of order 1: 1e-6)."""
    d = scenes.cube_medium(nder=1, res=8, spp=1, grid_res=4)
    sc = scenes.instantiate(gpu, d)
    v = np.concatenate([s.vertices for s in d.shapes]).astype(np.float64)
    base = np.cumsum([0] + [len(s.vertices) for s in d.shapes])
    f = np.concatenate([s.indices + base[i] for i, s in enumerate(d.shapes)])
    rays = []
    for x, y, z in itertools.product((-0.913, -0.237, 0.119, 0.771), repeat=3):
        for axis, sign, zero in itertools.product(range(3), (1.0, -1.0), (0.0, -0.0)):
            dirn = np.full(3, zero, np.float32)
            dirn[axis] = sign
            rays.append([x, y, z, *dirn, 1e-3, 1e30])
    rays = np.array(rays, np.float32)
    face, t = gpu.trace(sc, rays)
    want = _closest(v, f, rays)
    assert ((face >= 0) == np.isfinite(want)).all()
    hit = face >= 0
    assert hit.all()   # the enclosing sphere is behind everything
    assert np.abs(t[hit] - want[hit]).max() <= 1e-6 * want[hit].max()


@pytest.mark.parametrize("ntri", [1, 2, 3, 16, 17])
def test_smallest_trees_render_the_same_from_lds_and_hbm(gpu, ntri):
    """A single leaf under its wrapper node, two leaves, a leaf beside an inner node: a fan
    of emitting triangles seen directly. The image of the fan does not depend on where
    the tree is read from, and no stack entry runs into the tree's copy."""
    ang = np.linspace(0, 2.5, ntri + 1)
    v = np.concatenate([[[0, 0, 0]], np.stack([np.cos(ang), np.sin(ang), 0 * ang], -1)]).astype(np.float32)
    f = np.array([[0, k + 1, k + 2] for k in range(ntri)], np.int32)
    d = scenes.SceneDesc(nder=1, width=24, height=24, cam_to_world=scenes.look_at((0, 0.4, 3), (0, 0.4, 0), (0, 1, 0)),
                         cam_to_ndc=scenes.cam_to_ndc(45.0), shapes=[scenes.ShapeDesc(v, f, bsdf_id=0, light_id=0)],
                         bsdfs=[("diffuse", (0.5, 0.5, 0.5))], lights=[("area", 0, (3.0, 2.0, 1.0), True)], spp=64, max_bounces=2)
    sc = scenes.instantiate(gpu, d)
    lds = scenes.render_primal(gpu, d, seed=5, scene=sc)
    gpu.set_tree_in_hbm(sc, True)
    hbm = scenes.render_primal(gpu, d, seed=5, scene=sc)
    assert lds.max() == pytest.approx(3.0, rel=1e-6)
    assert np.allclose(lds, hbm, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("subdiv,rtol", [(3, 1e-5), (4, 1e-5)])
def test_middle_trees_render_the_same_from_lds_and_hbm(gpu, subdiv, rtol):
    """1,280 triangles fit in LDS once per compute unit, beside the stacks of one work-group of
    eight waves; 5,120 do not fit at all. Value and tangent images, child paths included,
    are the same from either memory (double sums in another order, rounded to float)."""
    d = scenes.ico_surface(nder=3, res=40, spp=32)
    v, f = scenes.icosphere(subdiv, 0.5, (0, 0.5, 0))
    vel = np.zeros((3, len(v), 3), np.float32)
    vel[0, :, 0] = vel[1, :, 1] = vel[2, :, 2] = 1.0
    d.shapes[1] = scenes.ShapeDesc(v, f, bsdf_id=1, velocities=vel)
    sc = scenes.instantiate(gpu, d)
    lds = scenes.render(gpu, d, seed=3, scene=sc, sppe=256).astype(np.float64)
    assert gpu.render_stats(sc)["children"] > 0
    gpu.set_tree_in_hbm(sc, True)
    hbm = scenes.render(gpu, d, seed=3, scene=sc, sppe=256).astype(np.float64)
    for lane in range(4):
        assert np.abs(lds[lane]).max() > 0
        assert np.allclose(lds[lane], hbm[lane], rtol=rtol, atol=rtol * 1e-2 * np.abs(lds[lane]).max()), lane


@pytest.mark.parametrize("subdiv", [2, 3, 4])
@pytest.mark.parametrize("kind", [1, 2, 3])
def test_primal_images_do_not_depend_on_where_the_tree_is(gpu, subdiv, kind):
    """320, 1,280 and 5,120 triangles: wholly in LDS for work-groups of four waves, of eight, and
    a prefix of the nodes only; against the tree in HBM alone. The same paths, each pixel's
    sum in another order (doubles rounded to float: 1e-6)."""
    d = scenes.ico_surface(nder=1, res=37, spp=5)
    v, f = scenes.icosphere(subdiv, 0.5, (0, 0.5, 0))
    d.shapes[1] = scenes.ShapeDesc(v, f, bsdf_id=1, velocities=np.zeros((1, len(v), 3), np.float32))
    sc = scenes.instantiate(gpu, d)
    a = scenes.render_primal(gpu, d, seed=9, scene=sc, kind=kind)
    gpu.set_tree_in_hbm(sc, True)
    b = scenes.render_primal(gpu, d, seed=9, scene=sc, kind=kind)
    assert a.max() > 0
    assert np.allclose(a, b, rtol=1e-6, atol=1e-9)
