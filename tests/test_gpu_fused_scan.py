"""The duplication scans for itself up to 2^21 Gaussians: the sizes around a block, around the size up to which the blend is queued ahead
of the number, and on both sides of the limit, passes after a first one, passes with fewer instances than expected and passes with more."""
import pytest
import torch

from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode, diff_rasterize, rasterize, update_max_weights
from htgs_amd.torch_bindings.rasterization import ScratchPool, run_max_weights

pytestmark = pytest.mark.gpu


# sums of a list's shares in another order: some 3e-7 times the root of its length
BOUND = 1e-5


def outgrown(counts, expected):
    """Whether a pass of so many instances had to make its lists again."""
    return expected != 0 and counts > expected + expected // 8 + 4096


@pytest.mark.parametrize("mode", [0, 3])
@pytest.mark.parametrize("n", [65_536, 65_537, 300_001, (1 << 21) - 1, 1 << 21, (1 << 21) + 1])
def test_passes_of_many_gaussians(cuda, n, mode):
    print(f"case n={n} mode={mode}", flush=True)
    scene = make_scene(1, n).to(cuda)
    scene.width, scene.height = 203, 149                     # a camera that looks at the middle of the cluster
    scene.VPM[0] += (scene.width / 2 - 640.0) * scene.VPM[3]
    scene.VPM[1] += (scene.height / 2 - 360.0) * scene.VPM[3]
    s = scene.settings(RasterizerMode(mode), 8)
    few = slice(0, n // 4)
    small = [t[few].contiguous() for t in scene.gaussians()]
    # (as many Gaussians, most of them out of sight: a pass of the same size with fewer instances)
    hidden = [scene.positions.clone(), *scene.gaussians()[1:]]
    hidden[0][n // 4:, 2] -= 1000.0
    want = {}
    for name, gaussians in (("all", scene.gaussians()), ("small", small), ("hidden", hidden)):
        fb = FrameBuffers(*gaussians, s, True, False, tight_lists=True)
        want[name] = (*(t.clone() for t in fb.run()), fb.n_instances)
        assert float(want[name][0].mean()) > 0.01
    inputs = {"all": scene.gaussians(), "small": small, "hidden": hidden}

    def check(name):
        expected = ScratchPool.current(cuda).expected((0, mode))
        image, depth = rasterize(*inputs[name], s, True, False)
        assert (image - want[name][0]).abs().max() < BOUND, name
        assert (depth.reshape(want[name][1].shape) - want[name][1]).abs().max() < 20.0 * BOUND, name
        return outgrown(want[name][2], expected)
    ScratchPool.clear()
    for name in ("all", "all", "small", "hidden", "all"):
        assert not check(name)
    # (a pool that expects few instances: the lists are made again)
    for name in ("small", "hidden"):
        ScratchPool.clear()
        assert not check(name) and not check(name)
        assert check("all")


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("n", [80_000, (1 << 21) - 255, (1 << 21) + 77])
def test_training_and_weights_of_many_gaussians(cuda, n, mode):
    """Around the limit, and around a frame that is queued behind its scan: gradients, whose rows are found through what the duplication
    leaves in the records, and weights against the stages, with and without the lists made a second time."""
    print(f"case n={n} mode={mode}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(5)
    scene = make_scene(0, 1000).to(cuda)
    seen = torch.rand(n, generator=g, device=cuda)
    positions = torch.rand(n, 3, generator=g, device=cuda) * 2.0 - 1.0
    rest = (torch.exp(torch.randn(n, 3, generator=g, device=cuda) * 0.5 - 4.0), torch.nn.functional.normalize(torch.randn(n, 4, generator=g, device=cuda)),
            torch.rand(n, 1, generator=g, device=cuda), torch.randn(n, 1, 3, generator=g, device=cuda), torch.zeros(n, 0, 3, device=cuda))
    up = torch.randn(3, scene.height, scene.width, generator=g, device=cuda)
    s = scene.settings(RasterizerMode(mode), 4)

    def view(shown):                                         # so many Gaussians in front of the camera, the others behind it
        p = positions.clone()
        p[:, 2] += torch.where(seen < shown / n, 4.0, -400.0)
        return p, *rest
    ScratchPool.clear()
    again = []
    for shown in (3000, 3000, 20_000, 20_000, 5000):
        gaussians = view(shown)
        expected = [ScratchPool.current(cuda).expected((what, mode)) for what in (1, 2)]
        leaves = [t.clone().requires_grad_() for t in gaussians]
        image = diff_rasterize(*leaves, torch.empty(0, device=cuda), s, False)
        fb = FrameBuffers(*gaussians, s, True, False, train=True, tight_lists=True, waves_per_tile=4)
        assert (image.detach() - fb.run_forward()).abs().max() < BOUND
        assert image.grad_fn.fb.frame.n_instances == fb.n_instances
        for a, b in zip(torch.autograd.grad(image, [t for t in leaves if t.numel()], up), fb.run_backward(up)):
            assert (a - b).norm() <= 1e-4 * b.norm()
        got, ref = torch.zeros(n, device=cuda), torch.zeros(n, device=cuda)
        update_max_weights(got, *gaussians[:4], s, 0.01)
        run_max_weights(ref, *gaussians[:4], s, 0.01)
        assert (got - ref).abs().max() < BOUND and float(got.max()) > 0.1
        again.append([outgrown(fb.n_instances, e) for e in expected])
    assert again[1:] == [[False, False], [True, True], [False, False], [False, False]]
