"""The staged AD kernels at the sizes where their lists, runs and batches can go wrong, and the
medium's tangents, which they sum over a segment before they meet the lanes."""
import numpy as np
import pytest
import torch

from dtrt_amd import scenes
from tests.helpers import assert_parity, renders

pytestmark = pytest.mark.gpu


def _furnace(nder, w, h, spp):
    v, f = scenes.icosphere(1, 5.0, inward=True)
    return scenes.SceneDesc(nder=nder, width=w, height=h, cam_to_world=scenes.look_at((0, 0, 0), (0, 0, 1), (0, 1, 0)),
                            cam_to_ndc=scenes.cam_to_ndc(60.0), shapes=[scenes.ShapeDesc(v, f, bsdf_id=0, light_id=0)],
                            bsdfs=[("diffuse", (0.0, 0.0, 0.0))], lights=[("area", 0, (1.0, 2.0, 0.5), True)], spp=spp,
                            max_bounces=3, sppe=0, sppse=0)


@pytest.mark.parametrize("nder,w,h,spp", [(1, 1, 1, 1), (1, 7, 5, 1), (3, 13, 9, 3), (1, 11, 3, 63), (3, 5, 3, 65), (8, 3, 2, 130),
                                          (2, 67, 41, 64)])
def test_every_sample_is_summed_into_its_pixel(gpu, nder, w, h, spp):
    """Camera inside a black sphere of constant emission: every sample sees exactly its
    radiance, so each pixel is that radiance whatever share of a wave its samples fill
    (sums of spp equal doubles, one float rounding: 1e-6)."""
    img = scenes.render(gpu, _furnace(nder, w, h, spp), seed=4)
    assert np.allclose(img[0], np.broadcast_to(np.float32([1.0, 2.0, 0.5]), img[0].shape), rtol=1e-6)
    assert (img[1:] == 0).all()


@pytest.mark.parametrize("nder,w,h,spp", [(3, 33, 17, 5), (1, 300, 201, 9)])
def test_batches_of_one_chunk_equal_one_batch(gpu, nder, w, h, spp):
    """The allocation-free render holds fewer samples in flight than the other (its path
    state is a share of the scratch area), so a chunk runs as several batches there.
    Same samples, same sums up to order (double sums rounded to float: 1e-5)."""
    d = scenes.cube_medium(nder=nder, res=64, spp=spp, grid_res=8)
    d.width, d.height = w, h
    sc = scenes.instantiate(gpu, d)
    opts = gpu.RenderOptions(3, spp, 6, 256, 4, True, -1, 0.0)
    a, b = torch.zeros(d.out_shape(), device="cuda"), torch.zeros(d.out_shape(), device="cuda")
    gpu.render_device(0, sc, opts, a.data_ptr())
    import ctypes as C
    st = opts._struct()
    fn = gpu.lib.dtrt_render_device_noalloc
    fn.argtypes = gpu.lib.dtrt_render_device.argtypes
    assert fn(0, sc._h, C.byref(st), b.data_ptr()) == 0
    torch.cuda.synchronize()
    assert float(a[0].max()) > 0
    for lane in range(nder + 1):
        assert torch.allclose(a[lane], b[lane], rtol=1e-5, atol=1e-7 * float(a[lane].abs().max()) + 1e-12), lane


def test_rotating_scaled_medium_matches_the_oracle(gpu, oracle):
    """Lanes that rotate the volume, move it and scale its density, in a medium that is
    itself placed by a rotation: every lane's image agrees with the oracle at 3 sigma."""
    d = scenes.cube_medium(nder=4, res=24, spp=16, grid_res=12)
    n = d.nder
    med = d.media[0]
    c, s = np.cos(0.4), np.sin(0.4)
    med.to_world = np.array([[c, 0, s, 0.05], [0, 1, 0, -0.02], [-s, 0, c, 0.03], [0, 0, 0, 1]], np.float32)
    med.trans_vel, med.rot_vel = np.zeros((n, 3), np.float32), np.zeros((n, 3), np.float32)
    med.d_scale = np.zeros(n, np.float32)
    med.rot_vel[0] = (0.3, 1.0, -0.2)
    med.trans_vel[1] = (0.5, -1.0, 0.25)
    med.d_scale[2] = 1.0
    med.rot_vel[3], med.trans_vel[3], med.d_scale[3] = (0.0, 0.4, 0.8), (0.2, 0.1, -0.6), 0.5
    for sh in d.shapes:
        sh.velocities = np.zeros((n, len(sh.vertices), 3), np.float32)
    kw = dict(mode=1 | 2 | 8, sppe=0, sppse=0)
    a = renders(gpu, d, range(1, 17), **kw)
    b = renders(oracle, d, range(101, 117), **kw)
    assert np.abs(a[:, 1:]).max() > 0
    assert_parity(a, b, 4, what="rotating medium")


def test_reflectance_lane_of_a_black_surface_matches_the_oracle(gpu, oracle):
    """A diffuse surface whose reflectance is zero but has a tangent: its light samples add
    nothing to the value and all of the lane's derivative, so they are not left out."""
    d = scenes.ico_surface(nder=2, res=24, spp=16)
    dref = np.zeros((2, 3), np.float32)
    dref[1] = (1.0, 0.5, 0.25)
    d.bsdfs[0] = ("diffuse", (0.0, 0.0, 0.0), dref)
    a = renders(gpu, d, range(1, 17), sppe=256)
    b = renders(oracle, d, range(101, 117), sppe=256)
    assert np.abs(a[:, 2]).max() > 0
    assert_parity(a, b, 4, what="black surface with a reflectance lane")


@pytest.mark.parametrize("nder,w,h,spp", [(1, 1, 1, 1), (1, 7, 5, 3), (8, 17, 13, 5), (3, 67, 41, 9), (1, 1024, 700, 7)])
def test_density_gradient_is_the_sum_of_its_pixels(gpu, nder, w, h, spp):
    """The adjoint's path lists leave out the samples of pixels without a gradient, so the
    gradient of all pixels, of every third one and of the others meet lists of every length
    (the largest case in two chunks). It is linear in the pixels and its paths do not
    depend on them, nor on the scene's lanes: the same samples added in another order
    (sums of up to 1e7 doubles, rounded to float and added once more in float: well
    within 1e-4 of the largest node)."""
    grads = {}
    for lanes in (1, nder):
        d = scenes.cube_medium(nder=lanes, res=64, spp=spp, grid_res=8)
        d.width, d.height = w, h
        sc = scenes.instantiate(gpu, d)
        opts = gpu.RenderOptions(5, spp, 6, 0, 0, True, 1 | 2 | 8)
        g = torch.as_tensor(np.random.default_rng(1).uniform(0.5, 1.5, size=(h, w, 3)).astype(np.float32), device="cuda")
        third = (torch.arange(h * w, device="cuda") % 3 == 0).view(h, w, 1)
        for name, part in (("all", g), ("third", g * third), ("rest", g * ~third), ("none", g * 0)):
            out = torch.zeros(d.media[0].density.shape, dtype=torch.float32, device="cuda")
            gpu.render_adjoint(sc, opts, 0, part.data_ptr(), out.data_ptr())
            torch.cuda.synchronize()
            grads[lanes, name] = out
    a = grads[1, "all"]
    tol = 1e-4 * float(a.abs().max())
    assert float((grads[1, "third"] + grads[1, "rest"] - a).abs().max()) <= tol
    assert float((grads[nder, "all"] - a).abs().max()) <= tol
    assert float(grads[1, "none"].abs().max()) == 0
    assert w * h * spp < 1000 or tol > 0
