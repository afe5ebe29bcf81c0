"""What a path keeps between bounces: the terms still to add and the medium it is in."""
import numpy as np
import pytest
import torch

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scene", ["medium", "surface"])
@pytest.mark.parametrize("mode", [0x7F, 0xFF, 0x3F | 1 << 9, 0x7FFFFFFF])
def test_mode_bits_that_name_no_term_are_ignored(gpu, scene, mode):
    """All six terms with further bits set, from a camera whose rays first scatter (inside the
    medium, before a diffuse surface): the image of mode -1, the same samples summed in
    another order (double sums rounded to float: 1e-6)."""
    if scene == "medium":
        d = scenes.cube_medium(nder=2, res=24, spp=8, grid_res=8)
        d.cam_to_world, d.cam_med = scenes.look_at((0.1, 0.05, 0.45), (0, 0, -0.2), (0, 1, 0)), 0
    else:
        d = scenes.ico_surface(nder=2, res=24, spp=8)
    sc = scenes.instantiate(gpu, d)
    kw = dict(seed=3, scene=sc, sppe=64)
    a, b = scenes.render(gpu, d, mode=-1, **kw), scenes.render(gpu, d, mode=mode, **kw)
    assert np.abs(a[0]).max() > 0 and np.abs(a[1]).max() > 0
    for lane in range(3):
        assert np.allclose(a[lane], b[lane], rtol=1e-6, atol=1e-8 * np.abs(a[lane]).max()), lane


@pytest.mark.parametrize("index", [253, 254, 255, 300, 5000])
def test_a_medium_of_any_index_is_found_again(gpu, index):
    """The cube's medium behind `index` others that no shape names: image and density gradient of
    the interior terms are those of the scene with that medium alone (sums in another
    order, rounded to float: 1e-6)."""
    def run(behind):
        d = scenes.cube_medium(nder=1, res=20, spp=8, grid_res=8)
        d.media = [scenes.MediumDesc("homogeneous", sigma_t=7.0)] * behind + d.media
        d.shapes[0].med_int = behind
        sc = scenes.instantiate(gpu, d)
        img = scenes.render(gpu, d, seed=5, scene=sc, mode=1 | 2 | 8, sppe=0, sppse=0)
        g = torch.ones((20, 20, 3), device="cuda")
        out = torch.zeros((8, 8, 8), device="cuda")
        gpu.render_adjoint(sc, gpu.RenderOptions(5, 8, d.max_bounces, 0, 0, True, 1 | 2 | 8), behind, g.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        return img, out.cpu().numpy()
    for a, b in zip(run(0), run(index)):
        assert np.abs(a).max() > 0
        assert np.allclose(a, b, rtol=1e-6, atol=1e-6 * np.abs(a).max())
