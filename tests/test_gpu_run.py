"""Whole passes by ``htgs_run``: a frame that is queued before the host knows its number of instances equals the frame taken
stage by stage, whether the number comes out as expected, larger (queued a second time), smaller or zero."""
import pytest
import torch

from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode, diff_rasterize, rasterize, update_max_weights
from htgs_amd.torch_bindings.rasterization import ScratchPool, run_max_weights

pytestmark = pytest.mark.gpu


def scenes(cuda):
    """few instances, many (more than the launches for the frame before were sized for), few again, none in view"""
    few, many = make_scene(0, 500).to(cuda), make_scene(0, 20_000).to(cuda)
    gone = make_scene(0, 700).to(cuda)
    gone.positions[:, 2] -= 100.0
    return few, many, few, gone, many


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
def test_render_equals_the_stages(cuda, mode):
    ScratchPool.clear()
    for i, scene in enumerate(scenes(cuda)):
        print(f"case mode={mode} frame={i}", flush=True)
        s = scene.settings(RasterizerMode(mode), 4)
        image, depth = rasterize(*scene.gaussians(), s, i % 2 == 0, False)
        want, want_depth = FrameBuffers(*scene.gaussians(), s, i % 2 == 0, False, tight_lists=True, waves_per_tile=4).run()
        assert torch.equal(image, want) and torch.equal(depth.reshape(want_depth.shape), want_depth)


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
def test_training_and_max_weights_equal_the_stages(cuda, mode):
    ScratchPool.clear()
    for i, scene in enumerate(scenes(cuda)):
        print(f"case mode={mode} frame={i}", flush=True)
        s = scene.settings(RasterizerMode(mode), 4)
        up = torch.randn(3, scene.height, scene.width, generator=torch.Generator().manual_seed(i)).to(cuda)
        leaves = [t.clone().requires_grad_() for t in scene.gaussians()]
        image = diff_rasterize(*leaves, torch.empty(0, device=cuda), s, False)
        grads = torch.autograd.grad(image, leaves, up)
        fb = FrameBuffers(*scene.gaussians(), s, True, False, train=True, tight_lists=True, waves_per_tile=4)
        assert torch.equal(image.detach(), fb.run_forward())
        for got, want in zip(grads, fb.run_backward(up)):
            assert torch.equal(got, want)
        n = scene.positions.shape[0]
        got, want = torch.zeros(n, device=cuda), torch.zeros(n, device=cuda)
        update_max_weights(got, *scene.gaussians()[:4], s, 0.01)
        run_max_weights(want, *scene.gaussians()[:4], s, 0.01)
        assert torch.equal(got, want)
