"""Two and four waves per tile (``htgs_frame.waves_per_tile``) against one: lists of less than a batch up to many, cores of every size,
pixels with fragments of exactly equal depth, the image-only path and the training pass."""
import pytest
import torch

from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode
from util import tie_scene

pytestmark = pytest.mark.gpu


def build(kind, cuda):
    scene = make_scene(1, {"thin": 2000, "dense": 300_000, "twins": 40_000}[kind])
    scene.width, scene.height = 203, 149                     # a camera that looks at the middle of the cluster
    scene.VPM[0] += (scene.width / 2 - 640.0) * scene.VPM[3]
    scene.VPM[1] += (scene.height / 2 - 360.0) * scene.VPM[3]
    if kind == "twins":                                      # three coincident copies of every Gaussian, of other colours and opacities
        for name in ("positions", "scales", "rotations", "sh_rest"):
            t = getattr(scene, name)
            setattr(scene, name, torch.cat([t, t, t]).contiguous())
        scene.sh_0 = torch.cat([scene.sh_0, -scene.sh_0, 0.5 * scene.sh_0]).contiguous()
        scene.opacities = torch.cat([scene.opacities, 0.7 * scene.opacities, 0.4 * scene.opacities]).contiguous()
    return scene.to(cuda)


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("K", [1, 2, 4, 8, 16, 32])
@pytest.mark.parametrize("mode", [0, 1, 3])
@pytest.mark.parametrize("kind", ["thin", "dense", "twins"])
def test_image_and_depth(cuda, kind, mode, K, fast):
    print(f"case kind={kind} mode={mode} K={K} fast={fast}", flush=True)
    if mode == 3 and K != 1:
        pytest.skip("no core")
    scene = build(kind, cuda)
    s = scene.settings(RasterizerMode(mode), K)
    for median, waves in ((False, 4), (True, 2)):
        one = FrameBuffers(*scene.gaussians(), s, True, median, fast=fast)
        four = FrameBuffers(*scene.gaussians(), s, True, median, fast=fast, waves_per_tile=waves)
        image, depth = one.run()
        image4, depth4 = four.run()
        longest = int((one.ranges[:, 1] - one.ranges[:, 0]).max())
        assert {"thin": longest < 64, "dense": longest > 300, "twins": longest > 128}[kind]
        if fast and kind == "twins":
            continue                                         # (which of two fragments of equal depth stays is open there)
        if mode == 1 and not fast and kind != "twins":       # (more of the twins' pixels are walked again, with alphas kept as floats)
            assert torch.equal(image4, image) and torch.equal(depth4, depth)
        else:
            assert (image4 - image).abs().max() < 2e-6
            assert fast or (depth4 - depth).abs().max() < 5e-5


@pytest.mark.parametrize("K,waves", [(1, 4), (4, 2), (16, 4), (32, 2)])
@pytest.mark.parametrize("mode", [0, 1, 3])
@pytest.mark.parametrize("kind", ["thin", "dense", "twins"])
def test_training_records(cuda, kind, mode, K, waves):
    print(f"case kind={kind} mode={mode} K={K}", flush=True)
    if mode == 3 and K != 1:
        pytest.skip("no core")
    scene = build(kind, cuda)
    s = scene.settings(RasterizerMode(mode), K)
    one = FrameBuffers(*scene.gaussians(), s, True, False, train=True)
    four = FrameBuffers(*scene.gaussians(), s, True, False, train=True, waves_per_tile=waves)
    a, b = one.run_forward(), four.run_forward()
    assert (a - b).abs().max() < 2e-6
    # (entries of pixels beyond the image are never written)
    if mode in (0, 1):
        assert torch.equal(one.records_in_image_order(one.core_idx), four.records_in_image_order(four.core_idx))
        x, y = one.records_in_image_order(one.core_info), four.records_in_image_order(four.core_info)
        assert (x - y).abs().max() < 1e-4 * max(1.0, float(x.abs().max()))
    if mode in (0, 3):
        x, y = one.records_in_image_order(one.tail_info), four.records_in_image_order(four.tail_info)
        assert ((x - y).abs() <= 1e-5 * (1.0 + x.abs())).all()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 64, 65, 127, 128, 129, 256, 257, 300, 513])
@pytest.mark.parametrize("mode", [0, 1, 3])
def test_shares(cuda, mode, n):
    """Lists of exactly n instances, around the lengths at which a wave more gets a batch, the batches grow or there is a round more:
    every instance is walked once.  Bounds as in test_image_and_depth."""
    g = torch.Generator().manual_seed(n)
    scene = tie_scene((2.0 + 30.0 * torch.rand(n, generator=g)).tolist(), (0.06 + 0.3 * torch.rand(n, generator=g)).tolist(), torch.rand(n, 3, generator=g).tolist()).to(cuda)
    for K in (4, 16) if mode != 3 else (1,):
        s = scene.settings(RasterizerMode(mode), K)
        one = FrameBuffers(*scene.gaussians(), s, True, False)
        image, depth = one.run()
        assert int((one.ranges[:, 1] - one.ranges[:, 0]).max()) == n
        trained = FrameBuffers(*scene.gaussians(), s, True, False, train=True).run_forward()
        for waves in (2, 4):
            print(f"case mode={mode} n={n} K={K} waves={waves}", flush=True)
            image4, depth4 = FrameBuffers(*scene.gaussians(), s, True, False, waves_per_tile=waves).run()
            assert (image4 - image).abs().max() < 2e-6 and (depth4 - depth).abs().max() < 5e-5
            assert (FrameBuffers(*scene.gaussians(), s, True, False, train=True, waves_per_tile=waves).run_forward() - trained).abs().max() < 2e-6
