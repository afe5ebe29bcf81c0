"""A step without the outputs that its caller may leave out."""
import pytest
import torch

from dtrt_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_lanes,with_loss", [(False, False), (True, False), (False, True)])
def test_a_step_without_loss_or_lanes_gives_the_other_outputs(gpu, with_lanes, with_loss):
    """Eager, captured and replayed: images and density gradient (and the output that is asked for)
    are those of the step with both, the same samples summed in another order (double
    sums rounded to float: 1e-6 of the largest entry)."""
    d = scenes.cube_medium(nder=2, res=16, spp=4, grid_res=8)
    sc = scenes.instantiate(gpu, d)
    fo = [gpu.RenderOptions(3, 4, 4, 64, 4, True, -1, 0.0)]
    ao = [gpu.RenderOptions(4, 4, 4, 0, 0, True, 1 | 2 | 8)]
    target = [torch.full((16, 16, 3), 0.25, device="cuda")]

    def outs():
        return ([torch.zeros((3, 16, 16, 3), device="cuda")], torch.zeros((8, 8, 8), device="cuda"),
                torch.zeros(2, dtype=torch.float64, device="cuda"), torch.zeros(1, dtype=torch.float64, device="cuda"))

    def same(got, want):
        torch.cuda.synchronize()
        for a, b in zip([*got[0], *got[1:]], [*want[0], *want[1:]]):
            if a is not None:
                assert float(b.abs().max()) > 0
                assert float((a - b).abs().max()) <= 1e-6 * float(b.abs().max())
    want = outs()
    gpu.step(sc, [None], fo, want[0], target, 0, ao, want[1], want[2], want[3])
    img, grad, lanes, loss = outs()
    got = img, grad, lanes if with_lanes else None, loss if with_loss else None
    gpu.step(sc, [None], fo, got[0], target, 0, ao, *got[1:])
    same(got, want)
    gpu.capture_step(sc, [None], fo, got[0], target, 0, ao, *got[1:])
    same(got, want)
    for _ in range(2):
        img[0].zero_(), grad.fill_(1.0)
        assert gpu.replay_step(sc, [3, 4]) == 0
        same(got, want)
