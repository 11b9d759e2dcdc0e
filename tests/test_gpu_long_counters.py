"""Work counters per die (``htgs_frame.long_counters``) and the shares that long lists are cut into with them: images, weights and
gradients against a frame that has neither, workgroups of sixteen waves (up to 512 Ki Gaussians) and of eight, and the counters
left as they were found."""
import ctypes

import numpy as np
import pytest
import torch

from htgs_amd import _native
from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode, rasterize, update_max_weights

pytestmark = pytest.mark.gpu
COUNTERS, SHARE = 288, 264


def scene_of(cuda, width, height, n, fat):
    scene = make_scene(1, n)
    scene.width, scene.height = width, height
    scene.VPM[0] += (width / 2 - 640.0) * scene.VPM[3]
    scene.VPM[1] += (height / 2 - 360.0) * scene.VPM[3]
    scene.scales = scene.scales * 2.0 ** fat
    return scene.to(cuda)


def with_counters(frame):
    frame.counters = torch.zeros(COUNTERS, dtype=torch.int32, device=frame.device)
    frame.frame.long_counters = frame.counters.data_ptr()
    return frame


def share_of(lengths, threshold):
    """half of what 4096 waves walk of the lists beyond the threshold's bin each (a list counts nine tenths of its bin's end)"""
    held = 0.0
    for n in lengths.tolist():
        p = n.bit_length() - 1
        end = ((5 + ((n >> (p - 2)) & 3)) << (p - 2)) - 1 if p >= 2 else 0
        held += 0.9 * end if end > threshold else 0.0
    return min(max(0.5 / 4096 * held, 128.0), float(threshold))


@pytest.mark.parametrize("mode,K", [(0, 4), (0, 32), (1, 16), (3, 1)])
@pytest.mark.parametrize("width,height,n,fat", [(512, 512, 100_000, 2.0), (520, 520, 60_000, 3.0), (328, 328, 524_289, 1.0)])
def test_image(cuda, mode, K, width, height, n, fat):
    print(f"case mode={mode} K={K} {width}x{height} n={n} fat={fat}", flush=True)
    scene = scene_of(cuda, width, height, n, fat)
    s = scene.settings(RasterizerMode(mode), K)
    image, _ = FrameBuffers(*scene.gaussians(), s, True, False).run()
    frame = with_counters(FrameBuffers(*scene.gaussians(), s, True, False, long_list_threshold=-1))
    got = frame.run()[0].clone()
    threshold, lengths = int(frame.long_tiles[5]), (frame.ranges[:, 1] - frame.ranges[:, 0]).cpu()
    assert int(lengths.max()) > threshold                    # (there are long lists)
    left = frame.counters.cpu()
    assert left[SHARE] == pytest.approx(share_of(lengths, threshold), rel=1e-3, abs=1.0)
    left[SHARE] = 0
    assert int(left.abs().sum()) == 0 and int(frame.long_tiles[:5].abs().sum()) == 0
    assert (got - image).abs().max() < 3e-6                  # (sums in another order)
    frame.blend()                                            # (the list is empty again)
    assert torch.equal(frame.image, got)
    assert (rasterize(*scene.gaussians(), s, True, False)[0] - image).abs().max() < 3e-6


@pytest.mark.parametrize("mode,K", [(0, 16), (1, 4), (3, 1)])
def test_training(cuda, mode, K):
    print(f"case mode={mode} K={K}", flush=True)
    scene = scene_of(cuda, 520, 520, 60_000, 3.0)
    s = scene.settings(RasterizerMode(mode), K)
    grad = torch.randn(3, 520, 520, device=cuda, generator=torch.Generator(device=cuda).manual_seed(3))
    one = FrameBuffers(*scene.gaussians(), s, True, False, train=True)
    image, grads = one.run_forward(), [g.clone() for g in one.run_backward(grad)]
    frame = with_counters(FrameBuffers(*scene.gaussians(), s, True, False, train=True, long_list_threshold=-1))
    assert (frame.run_forward() - image).abs().max() < 3e-6
    assert int((frame.ranges[:, 1] - frame.ranges[:, 0]).max()) > int(frame.long_tiles[5])
    for a, b in zip(frame.run_backward(grad), grads):        # (float32 sums over the pixels in the same order, of tails summed in another)
        assert (a - b).norm() <= 1e-4 * b.norm()
    left = frame.counters.cpu()
    left[SHARE] = 0
    assert int(left.abs().sum()) == 0


@pytest.mark.parametrize("mode,K", [(0, 16), (1, 4), (3, 1)])
def test_max_weights(cuda, mode, K):
    print(f"case mode={mode} K={K}", flush=True)
    scene = scene_of(cuda, 328, 328, 200_000, 2.0)
    s = scene.settings(RasterizerMode(mode), K)
    got, ref = (torch.zeros(200_000, device=cuda) for _ in range(2))
    g = scene.gaussians()
    update_max_weights(got, *g[:4], s, 0.02)
    frame = FrameBuffers(*g[:4], None, None, s, True, False)
    frame.long_tiles = None
    frame.frame.long_tiles = 0                               # (one wave per tile)
    _native.check(frame.lib.htgs_max_weights_front(ctypes.byref(frame.frame)))
    frame.alloc_instances(frame.read_instance_count())
    _native.check(frame.lib.htgs_max_weights_back(ctypes.byref(frame.frame), ref.data_ptr(), 0.02))
    # (weights are products: only the tail's share depends on an order of sums; one at the threshold may fall on either side)
    a, b = got.cpu().numpy(), ref.cpu().numpy()
    both = (a > 0) & (b > 0)
    assert both.sum() > 50 and ((a > 0) != (b > 0)).sum() <= 2
    np.testing.assert_allclose(a[both], b[both], rtol=1e-5)
