"""Trees in HBM, on both sides of the lines between the kernels for few paths and for many:
the same paths as with the tree in LDS, summed in another order (doubles rounded to float)."""
import numpy as np
import pytest

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu


def _surface(gpu, nder, res, spp):
    d = scenes.ico_surface(nder=nder, res=res, spp=spp)
    v, f = scenes.icosphere(2, 0.5, (0, 0.5, 0))
    vel = np.zeros((nder, len(v), 3), np.float32)
    vel[0, :, 0] = 1.0
    d.shapes[1] = scenes.ShapeDesc(v, f, bsdf_id=1, velocities=vel)
    return d, scenes.instantiate(gpu, d)


@pytest.mark.parametrize("kind", [1, 2, 3])
@pytest.mark.parametrize("res,spp", [(64, 32), (65, 32), (128, 10), (3, 1)])
def test_primal_samples_around_two_waves_per_simd(gpu, kind, res, spp):
    """131,072 samples fill two waves per SIMD exactly; 135,200 and 163,840 do not fit."""
    d, sc = _surface(gpu, 1, res, spp)
    lds = scenes.render_primal(gpu, d, seed=9, scene=sc, kind=kind)
    gpu.set_tree_in_hbm(sc, True)
    hbm = scenes.render_primal(gpu, d, seed=9, scene=sc, kind=kind)
    assert lds.max() > 0
    assert np.allclose(lds, hbm, rtol=1e-6, atol=1e-9)


@pytest.mark.parametrize("integrator", ["volpath", "path"])
@pytest.mark.parametrize("nder,sppe", [(1, 200), (1, 60000), (3, 60000), (8, 60000)])
def test_child_queues_of_either_length(gpu, integrator, nder, sppe):
    """Up to 50,000 records per bounce of the limit (2) and far more of them."""
    d, sc = _surface(gpu, nder, 24, 4)
    kw = dict(seed=3, scene=sc, sppe=sppe, max_bounces=2, integrator=gpu.VolPathTracerAD() if integrator == "volpath" else gpu.PathTracerAD())
    lds = scenes.render(gpu, d, **kw).astype(np.float64)
    children = gpu.render_stats(sc)["children"]
    assert (children > 200000) == (sppe > 200) and children > 0
    gpu.set_tree_in_hbm(sc, True)
    hbm = scenes.render(gpu, d, **kw).astype(np.float64)
    assert np.abs(lds[1]).max() > 0
    for lane in range(nder + 1):
        assert np.allclose(lds[lane], hbm[lane], rtol=1e-5, atol=1e-7 * np.abs(lds[lane]).max()), lane


@pytest.mark.parametrize("nder,sppe", [(1, 200), (3, 60000)])
def test_direct_child_queues_do_not_depend_on_the_limit(gpu, nder, sppe):
    """DirectAD's children have one bounce: a limit of 50 gives the images of a limit of 2, in either kernel."""
    d, sc = _surface(gpu, nder, 24, 4)
    kw = dict(seed=3, scene=sc, sppe=sppe, integrator=gpu.DirectAD())
    lds = scenes.render(gpu, d, max_bounces=2, **kw).astype(np.float64)
    assert gpu.render_stats(sc)["children"] > 0
    gpu.set_tree_in_hbm(sc, True)
    assert np.abs(lds[1]).max() > 0
    for limit in (2, 50):
        hbm = scenes.render(gpu, d, max_bounces=limit, **kw).astype(np.float64)
        for lane in range(nder + 1):
            assert np.allclose(lds[lane], hbm[lane], rtol=1e-5, atol=1e-7 * np.abs(lds[lane]).max()), (limit, lane)
