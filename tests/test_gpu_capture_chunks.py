"""Captured schedules where the child queue holds what 64K samples push, but not what 256K do."""
import numpy as np
import pytest
import torch

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu

RECORD = 144   # bytes of a child record of one lane in double


def _dense(gpu):
    """An evenly filled image (the middle of the cube), 327,680 samples of it, and a queue for 1.6 times
    what 64K of them push: four times 64K overflow it, and so do not the chunks that
    follow a first one of 64K, which aim at three quarters of it."""
    d = scenes.cube_medium(nder=1, res=768, spp=5, grid_res=8, crop=(256, 256, 256, 256))
    sc = scenes.instantiate(gpu, d)
    opts = gpu.RenderOptions(3, 5, 4, 0, 10, True, -1, 0.0)
    img = torch.zeros((2, 256, 256, 3), device="cuda")
    gpu.render_views(sc, [None], [opts], [img])
    st = gpu.render_stats(sc)
    gpu.set_queue_budget(sc, int(1.6 * 65536 * st["children"] / st["ad_samples"]) * RECORD)
    return sc, opts


def _same(a, b):
    assert float(a.abs().max()) > 0
    for lane in range(len(a)):
        assert torch.allclose(a[lane], b[lane], rtol=1e-6, atol=1e-8 * float(a[lane].abs().max())), lane


def test_views_with_a_dense_first_chunk_are_captured(gpu):
    """The capture is accepted, leaves the eager image, and a replay of another seed is that
    seed's eager render (the same samples summed in another order: 1e-6)."""
    sc, opts = _dense(gpu)
    want = {}
    for seed in (3, 11):
        o = gpu.RenderOptions(seed, 5, 4, 0, 10, True, -1, 0.0)
        want[seed] = torch.zeros((2, 256, 256, 3), device="cuda")
        gpu.render_views(sc, [None], [o], [want[seed]])
    img = torch.zeros((2, 256, 256, 3), device="cuda")
    gpu.capture_views(sc, [None], [opts], [img])
    torch.cuda.synchronize()
    _same(img, want[3])
    for seed in (11, 3, 11):
        assert gpu.replay_views(sc, [seed]) == 0
        torch.cuda.synchronize()
        _same(img, want[seed])


def test_a_step_with_a_dense_first_chunk_is_captured(gpu):
    sc, opts = _dense(gpu)
    adj = gpu.RenderOptions(4, 2, 4, 0, 0, True, 1 | 2 | 8)
    cam = scenes.cube_medium(nder=1, res=768, spp=5, grid_res=8)
    camera = gpu.Camera(768, 768, np.ascontiguousarray(cam.cam_to_world, np.float32), np.ascontiguousarray(cam.cam_to_ndc, np.float32),
                        1e-2, -1, None)
    camera.set_rect(256, 256, 256, 256)
    target = torch.zeros((256, 256, 3), device="cuda")
    img, grad = torch.zeros((2, 256, 256, 3), device="cuda"), torch.zeros((8, 8, 8), device="cuda")
    loss = torch.zeros(1, dtype=torch.float64, device="cuda")
    gpu.step(sc, [camera], [opts], [img], [target], 0, [adj], grad, None, loss)
    torch.cuda.synchronize()
    want = img.clone(), grad.clone()
    gpu.capture_step(sc, [camera], [opts], [img], [target], 0, [adj], grad, None, loss)
    for _ in range(2):
        img.zero_(), grad.zero_()
        assert gpu.replay_step(sc, [3, 4]) == 0
        torch.cuda.synchronize()
        _same(want[0], img)
        assert torch.allclose(want[1], grad, rtol=1e-5, atol=1e-6 * float(want[1].abs().max()))
