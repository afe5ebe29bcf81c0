"""Samples as batches, lists that run to their ends in one launch, and bounce limits far above
the paths' lengths: the same samples whichever way they run, summed in another order
(doubles rounded to float: 1e-6)."""
import numpy as np
import pytest
import torch

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu


def _same(a, b):
    a, b = a.double(), b.double()
    assert float(a[0].abs().max()) > 0
    for lane in range(len(a)):
        assert float((a[lane] - b[lane]).abs().max()) <= 1e-6 * float(b[lane].abs().max()), lane


def _render(gpu, sc, d, opts):
    img = torch.zeros(d.out_shape(), device="cuda")
    gpu.render_device(0, sc, opts, img.data_ptr())
    torch.cuda.synchronize()
    return img


def _scene(gpu, kind, nder):
    if kind == "cube":
        d = scenes.cube_medium(nder=nder, res=24, spp=7, grid_res=8)
        d.height = 19
    else:
        d = scenes.dielectric_medium(nder=nder, res=18, spp=5, freq=6, grid_res=8)
    return d, scenes.instantiate(gpu, d)


@pytest.mark.parametrize("kind,nder,depth", [("cube", 1, 6), ("cube", 3, 6), ("dielectric", 8, 6), ("cube", 2, 40), ("dielectric", 3, 200),
                                             ("cube", 16, 0), ("cube", 1, 1)])
def test_batches_and_tails_give_the_same_image(gpu, kind, nder, depth):
    """Batches of 64 and 192 samples (a partial last one), and tails of none, one path, a few waves and
    every path, against one batch that runs bounce by bounce; then all of it with a child
    queue so small that replay lists span batches too."""
    d, sc = _scene(gpu, kind, nder)
    opts = gpu.RenderOptions(3, d.spp, depth, 64, 4, True, -1, 0.0)
    gpu.set_ad_batch(sc, 0, 0)
    want = _render(gpu, sc, d, opts)
    settings = [(64, 0), (192, 0), (0, 1), (0, 100), (0, 1 << 20), (192, 33), (192, 192)]
    for slots, tail in settings:
        gpu.set_ad_batch(sc, slots, tail)
        _same(_render(gpu, sc, d, opts), want)
    if depth in (6, 40):
        gpu.set_queue_budget(sc, 16 << 10)
        for slots, tail in [(0, 0), (64, 0), (192, 100), (0, -1)]:
            gpu.set_ad_batch(sc, slots, tail)
            _same(_render(gpu, sc, d, opts), want)
            assert gpu.render_stats(sc)["replayed"] > 192


@pytest.mark.parametrize("nder,depth", [(1, 6), (8, 6), (2, 40), (1, 200), (1, 2)])
def test_batches_and_tails_give_the_same_density_gradient(gpu, nder, depth):
    d, sc = _scene(gpu, "cube", nder)
    opts = gpu.RenderOptions(5, d.spp, depth, 0, 0, True, 1 | 2 | 8)
    g = torch.as_tensor(np.random.default_rng(2).normal(size=(d.height, d.width, 3)).astype(np.float32), device="cuda")
    g[::3] = 0   # rows whose samples take no part
    grads = []
    for slots, tail in [(0, 0), (64, 0), (192, 0), (0, 1), (0, 100), (0, -1), (192, 50)]:
        gpu.set_ad_batch(sc, slots, tail)
        out = torch.zeros(d.media[0].density.shape, device="cuda")
        gpu.render_adjoint(sc, opts, 0, g.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        grads.append(out)
        _same(out[None], grads[0][None])


@pytest.mark.parametrize("tail", [0, -1])
def test_a_graph_replays_the_same_at_a_high_limit(gpu, tail):
    """Captured launches go up to the limit, eager ones end with the paths."""
    d, sc = _scene(gpu, "cube", 1)
    gpu.set_ad_batch(sc, 0, tail)
    opts = [gpu.RenderOptions(s, d.spp, 100, 64, 4, True, -1, 0.0) for s in (3, 9)]
    want = [_render(gpu, sc, d, o) for o in opts]
    img = torch.zeros(d.out_shape(), device="cuda")
    gpu.capture_views(sc, [None], [opts[0]], [img])
    for k in (1, 0, 1):
        assert gpu.replay_views(sc, [(3, 9)[k]]) == 0
        torch.cuda.synchronize()
        _same(img, want[k])


def test_path_state_for_fewer_samples_where_memory_is_short(gpu):
    """Four batches instead of one when only 70,000 samples' state can be had; an error, and no
    image, when not even 64K can."""
    d = scenes.cube_medium(nder=1, res=256, spp=3, grid_res=8)
    opts = gpu.RenderOptions(3, 3, 4, 64, 4, True, -1, 0.0)
    want = _render(gpu, scenes.instantiate(gpu, d), d, opts)
    sc = scenes.instantiate(gpu, d)
    gpu.set_ad_batch(sc, 0, -1, 70000)
    _same(_render(gpu, sc, d, opts), want)
    sc = scenes.instantiate(gpu, d)
    gpu.set_ad_batch(sc, 0, -1, 40000)
    img = torch.zeros(d.out_shape(), device="cuda")
    with pytest.raises(RuntimeError):
        gpu.render_device(0, sc, opts, img.data_ptr())
    assert float(img.abs().max()) == 0
    gpu.set_ad_batch(sc)
    _same(_render(gpu, sc, d, opts), want)


def test_a_larger_adjoint_keeps_a_captured_step_alive(gpu):
    """The step's path state is not taken away by an eager adjoint of 800 times its samples, which
    runs in as many batches as its own size asks for."""
    d, sc = _scene(gpu, "cube", 1)
    fo = [gpu.RenderOptions(3, 2, 4, 64, 4, True, -1, 0.0)]
    ao = [gpu.RenderOptions(4, 2, 4, 0, 0, True, 1 | 2 | 8)]
    big = gpu.RenderOptions(6, 1600, 4, 0, 0, True, 1 | 2 | 8)
    g = torch.ones((d.height, d.width, 3), device="cuda")

    def adjoint(scene):
        out = torch.zeros((8, 8, 8), device="cuda")
        gpu.render_adjoint(scene, big, 0, g.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        return out
    want = adjoint(scenes.instantiate(gpu, d))
    img, target = torch.zeros(d.out_shape(), device="cuda"), torch.zeros((d.height, d.width, 3), device="cuda")
    grad, loss = torch.zeros((8, 8, 8), device="cuda"), torch.zeros(1, dtype=torch.float64, device="cuda")
    gpu.capture_step(sc, [None], fo, [img], [target], 0, ao, grad, None, loss)
    torch.cuda.synchronize()
    step = img.clone(), grad.clone()
    _same(adjoint(sc)[None], want[None])
    for _ in range(2):
        img.zero_(), grad.zero_()
        assert gpu.replay_step(sc, [3, 4]) == 0
        torch.cuda.synchronize()
        _same(img, step[0])
        _same(grad[None], step[1][None])
    _same(adjoint(sc)[None], want[None])
