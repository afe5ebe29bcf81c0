"""The autotuner leaves alone what the integrator's kernels do not read."""
import pytest

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before", [64, 128, 256])
def test_the_ad_work_group_is_tuned_for_the_integrators_that_have_one(gpu, before):
    d = scenes.ico_surface(nder=1, res=32, spp=4)
    sc = scenes.instantiate(gpu, d)
    opts = gpu.RenderOptions(3, 4, 3, 64, 4, True, -1, 0.0)
    gpu.set_launch_settings(sc, ad_workgroup=before)
    _, st = gpu.autotune(sc, opts, integrator=0)
    assert st["ad_workgroup"] == before
    _, st = gpu.autotune(sc, opts, integrator=6)
    assert st["ad_workgroup"] in (64, 128, 256)
