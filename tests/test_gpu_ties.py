"""The HIP kernels against the hand-computed pixels of tests/test_oracle_ties.py (no oracle in between): fragments of
exactly equal depth in HYBRID_BLEND's core must come out in the order of the reference's exchange walk
(R/include/hybrid_blend/kernels/inference.cuh:159-167) -- through the kernel with one wave per tile (threshold 0, the
default of 8192: the core as sorted keys, pairs settled from it, three of a depth walked a second time; threshold 2^31 - 1: the
exchange insertion throughout), through the kernels that share a long list between waves (threshold forced down to 2
instances: the cores are merged and three of a depth get the second look), through the kernels of two and four waves a tile, and in the
core indices the training pass records."""
import numpy as np
import pytest
import torch

from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode
from test_oracle_ties import PX, THREE, TWO, exchange_walk
from util import hybrid_pixel_by_hand, tie_scene, u32

pytestmark = pytest.mark.gpu

CASES = [(TWO, [4, 0, 2, 1], [3]), (THREE, [4, 0, 2, 3], [1])]


@pytest.mark.parametrize("case,core,tail", CASES)
@pytest.mark.parametrize("threshold", [0, 2, 2 ** 31 - 1])
def test_inference_pixel_with_equal_depths(cuda, case, core, tail, threshold):
    print(f"case depths={case['depths']} threshold={threshold}", flush=True)
    scene = tie_scene(**case).to(cuda)
    fb = FrameBuffers(*scene.gaussians(), scene.settings(RasterizerMode.HYBRID_BLEND, 4), True, False, long_list_threshold=threshold)
    image, depth = fb.run()
    torch.cuda.synchronize()
    want_rgb, want_depth = hybrid_pixel_by_hand(core, tail, case["depths"], case["opacities"], case["colours"])
    assert np.abs(image[:, PX, PX].cpu().numpy() - want_rgb).max() <= 2e-6
    assert abs(float(depth[PX, PX]) - want_depth) <= 1e-5 * want_depth


@pytest.mark.parametrize("case,core,tail", CASES)
@pytest.mark.parametrize("threshold", [0, 2])
def test_recorded_core_with_equal_depths(cuda, case, core, tail, threshold):
    print(f"case depths={case['depths']} threshold={threshold}", flush=True)
    scene = tie_scene(**case).to(cuda)
    fb = FrameBuffers(*scene.gaussians(), scene.settings(RasterizerMode.HYBRID_BLEND, 4), True, False, train=True, long_list_threshold=threshold)
    fb.run_forward()
    torch.cuda.synchronize()
    idx = u32(fb.records_in_image_order(fb.core_idx))[:, PX * scene.width + PX]
    assert idx.tolist() == core


# What each wave has first: (depth, opacity); its share is filled up behind it.  Depths that are round numbers are alike in the lower half of
# their bit patterns, whatever note of an earlier tie a wave has kept.
EARLIER = [(1.0, 0.2), (1.25, 0.2), (1.5, 0.2), (4.0, 0.2), (4.0, 0.3), (3.0, 0.2)]
ROUND = {
    "a pair of another wave's": [EARLIER, [(2.0, 0.3), (2.0, 0.1)]],
    "one of each wave's": [EARLIER[:5] + [(2.0, 0.3)], [(2.0, 0.1)]],
    "a pair of the last wave's": [EARLIER, [], [(8.0, 0.2), (8.0, 0.2)], [(2.0, 0.3), (2.0, 0.1)]],
    "one of each of the last waves'": [EARLIER, EARLIER[3:], [(2.0, 0.3)], [(2.0, 0.1)]],
}


def pixel(scene, mode, K, waves, threshold=0):
    fb = FrameBuffers(*scene.gaussians(), scene.settings(RasterizerMode(mode), K), True, False, waves_per_tile=waves, long_list_threshold=threshold)
    image, depth = fb.run()
    return image[:, PX, PX].cpu().numpy(), float(depth[PX, PX])


@pytest.mark.parametrize("arrangement", ROUND)
@pytest.mark.parametrize("mode", [0, 1])
def test_ties_of_round_depths_between_waves(cuda, mode, arrangement):
    shares, per = ROUND[arrangement], 8 if mode == 0 else 16
    fragments = [f for share in shares for f in share + [(8.0 + 0.25 * k, 0.2) for k in range(per - len(share))]]
    depths, opacities = [list(v) for v in zip(*fragments)]
    colours = torch.rand(len(depths), 3, generator=torch.Generator().manual_seed(1)).tolist()
    core, tail = exchange_walk(list(zip(depths, range(len(depths)))), 4)
    first = depths.index(2.0)
    assert core[3] == first                                     # the more opaque of the two
    want_rgb, want_depth = hybrid_pixel_by_hand(core, tail if mode == 0 else [], depths, opacities, colours)
    scene = tie_scene(depths, opacities, colours).to(cuda)
    for waves in (1, len(shares)):
        print(f"case mode={mode} arrangement={arrangement} waves={waves}", flush=True)
        rgb, depth = pixel(scene, mode, 4, waves)
        assert np.abs(rgb - want_rgb).max() <= 4e-6 and abs(depth - want_depth) <= 1e-5 * want_depth


@pytest.mark.parametrize("K", [1, 2, 4, 8])
@pytest.mark.parametrize("mode", [0, 1])
def test_many_ties_of_round_depths(cuda, mode, K):
    """Lists whose depths are a few round numbers, every pixel with ties of two, three and more wherever they fall among the waves' shares."""
    g = torch.Generator().manual_seed(7)
    steps = torch.tensor([0.5, 1.0, 1.25, 1.5, 2.0, 2.5, 3.0, 4.0, 5.0, 6.0, 7.0, 8.0, 10.0, 12.0, 14.0, 16.0, 20.0, 24.0, 28.0, 32.0])
    for n in (16, 24, 32, 48, 64, 96):
        for _ in range(6):
            depths = steps[torch.randint(len(steps), (n,), generator=g)].tolist()
            opacities, colours = (0.06 + 0.3 * torch.rand(n, generator=g)).tolist(), torch.rand(n, 3, generator=g).tolist()
            core, tail = exchange_walk(list(zip(depths, range(n))), K)
            want_rgb, want_depth = hybrid_pixel_by_hand(core, tail if mode == 0 else [], depths, opacities, colours)
            scene = tie_scene(depths, opacities, colours).to(cuda)
            for waves in (1, 2, 4):
                print(f"case mode={mode} K={K} n={n} waves={waves}", flush=True)
                rgb, depth = pixel(scene, mode, K, waves)
                assert np.abs(rgb - want_rgb).max() <= 4e-6 and abs(depth - want_depth) <= 1e-5 * want_depth
