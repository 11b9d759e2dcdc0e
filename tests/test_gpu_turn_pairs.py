"""The inference walks take two turns of a batch at a time; a batch with an odd number of turns ends with a turn of dummy slots.  Lists
around a batch's 64 entries, odd and even, against the CPU oracle, and against the walk of one turn at a time with the core as
floats (HYBRID_BLEND, ALPHA_BLEND_FIRST_K)."""
import numpy as np
import pytest
import torch

from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode
from util import oracle_render, tie_scene

pytestmark = pytest.mark.gpu

TOL = 1e-4
# alphas held as fractions of 23 bits (2^-24 each) in a core of at most 32, and sums in the same order
BETWEEN = 1e-5


@pytest.mark.parametrize("waves", [0, 2])
@pytest.mark.parametrize("mode,K", [(0, 2), (0, 16), (0, 32), (1, 4), (1, 16), (3, 1)])
@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 127, 129])
def test_lists_around_a_batch(cuda, n, mode, K, waves):
    print(f"case n={n} mode={mode} K={K} waves={waves}", flush=True)
    rng = np.random.default_rng(n)
    scene = tie_scene(rng.uniform(1.0, 9.0, n).tolist(), rng.uniform(0.02, 1.0, n).tolist(), rng.uniform(0.0, 1.0, (n, 3)).tolist())
    ref = oracle_render(scene, mode, K)
    gpu = scene.to(cuda)
    s = gpu.settings(RasterizerMode(mode), K)
    fb = FrameBuffers(*gpu.gaussians(), s, True, False, waves_per_tile=waves)
    image, depth = (t.cpu().numpy() for t in fb.run())
    assert int((fb.ranges[:, 1] - fb.ranges[:, 0]).max()) == n and ref["image"].max() > 0.01
    assert np.abs(image - ref["image"]).max() <= TOL and np.abs(depth - ref["depth"]).max() <= TOL
    plain, plain_depth = FrameBuffers(*gpu.gaussians(), s, True, False, long_list_threshold=2 ** 31 - 1).run()
    assert np.abs(image - plain.cpu().numpy()).max() <= BETWEEN and np.abs(depth - plain_depth.cpu().numpy()).max() <= 10.0 * BETWEEN
    fast = FrameBuffers(*gpu.gaussians(), s, True, False, fast=True, waves_per_tile=waves).run()[0]
    assert np.abs(fast.cpu().numpy() - ref["image"]).max() <= 1e-3


@pytest.mark.parametrize("scale", [1e-8, 1e-10, 1e-11, 3e-12])
@pytest.mark.parametrize("mode", [0, 1, 3])
def test_a_direction_outside_the_refined_reciprocal(cuda, mode, scale):
    """|d|^2 (it goes with the fourth power of the scale) below 2^-120 at one Gaussian of three, at the one pixel it reaches: both
    turns take the division, and the other Gaussians' fragments come out as they do beside an ordinary one."""
    scene = tie_scene([2.0, 3.0, 4.0], [0.5, 0.6, 0.7], [[0.9, 0.1, 0.1], [0.1, 0.9, 0.1], [0.1, 0.1, 0.9]])
    scene.scales[1] = scale
    ref = oracle_render(scene, mode, 4)
    gpu = scene.to(cuda)
    image, depth = FrameBuffers(*gpu.gaussians(), gpu.settings(RasterizerMode(mode), 4), True, False).run()
    torch.cuda.synchronize()
    np.testing.assert_allclose(image.cpu().numpy(), ref["image"], rtol=0, atol=TOL, equal_nan=True)
    np.testing.assert_allclose(depth.cpu().numpy(), ref["depth"], rtol=0, atol=TOL, equal_nan=True)
