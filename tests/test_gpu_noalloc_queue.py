"""The scratch area of the allocation-free render, as far as each integrator needs it."""
import ctypes as C

import pytest
import torch

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [6, 0])
def test_children_that_fit_the_scratch_area_are_not_replayed(gpu, kind):
    """The 256 MiB hold 1.86M records of one lane in double. PathTracerAD keeps no path state there, so
    1.6M of them fit beside the small image; VolPathTracerAD keeps 13M for 35K samples (364 bytes each),
    not a quarter of the area. The image is that of the other render (sums in another order,
    rounded to float: 1e-6 of each lane's largest entry)."""
    d = scenes.ico_surface(nder=1, res=32, spp=8)
    sc = scenes.instantiate(gpu, d)
    per = {}
    for sppse in (400,):
        o = gpu.RenderOptions(3, 4, 3, 0, sppse, True, -1, 0.0)
        img = torch.zeros(d.out_shape(), device="cuda")
        gpu.render_device(kind, sc, o, img.data_ptr())
        st = gpu.render_stats(sc)
        per[sppse] = st["children"] / st["ad_samples"]
    spp = int(1.6e6 / (per[400] * 32 * 32))
    assert 4 <= spp <= 256
    o = gpu.RenderOptions(3, spp, 3, 0, 400, True, -1, 0.0)
    a, b = torch.zeros(d.out_shape(), device="cuda"), torch.zeros(d.out_shape(), device="cuda")
    gpu.render_device(kind, sc, o, a.data_ptr())
    st = o._struct()
    fn = gpu.lib.dtrt_render_device_noalloc
    fn.argtypes = gpu.lib.dtrt_render_device.argtypes
    assert fn(kind, sc._h, C.byref(st), b.data_ptr()) == 0
    torch.cuda.synchronize()
    stats = gpu.render_stats(sc)
    assert 1.4e6 < stats["children"] < 1.75e6 and stats["replayed"] == 0
    for lane in range(2):
        assert float(a[lane].abs().max()) > 0
        assert float((a[lane] - b[lane]).abs().max()) <= 1e-6 * float(a[lane].abs().max()), lane
