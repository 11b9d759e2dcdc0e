"""The list length that htgs_extract_ranges chooses (``long_list_threshold`` < 0): its value against the lengths of the lists, for
grids below and above the size of the one-workgroup tile order and with few instances and many, and the images with it."""
import pytest
import torch

from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode

pytestmark = pytest.mark.gpu


def chosen(lengths, waves):
    """the longest of the bins' upper ends (four bins per power of two) that 1.5 times the turns of a launch over the lists up to it allow"""
    best, held = 512, 0.0
    counts = {}
    for n in lengths.tolist():
        if n > 0:
            p = n.bit_length() - 1
            end = ((5 + ((n >> (p - 2)) & 3)) << (p - 2)) - 1 if p >= 2 else (1 << (p + 1)) - 1
            counts[end] = counts.get(end, 0) + 1
    ends = sorted(set(counts) | {((5 + sub) << (p - 2)) - 1 for p in range(2, 13) for sub in range(4)})
    for end in ends:
        held += counts.get(end, 0) * 0.9 * end
        if end <= 8192 and end <= 1.5 / 5120 * waves * held:
            best = max(best, end)
    return best


@pytest.mark.parametrize("mode,K", [(0, 4), (0, 32), (1, 16), (3, 1)])
@pytest.mark.parametrize("width,height,n,fat,waves", [(203, 149, 3000, 0.0, 4), (512, 512, 100_000, 2.0, 4), (520, 512, 100_000, 2.0, 2), (520, 520, 60_000, 3.0, 1)])
def test_threshold_and_image(cuda, mode, K, width, height, n, fat, waves):
    print(f"case mode={mode} K={K} {width}x{height} n={n} fat={fat} waves={waves}", flush=True)
    scene = make_scene(1, n)
    scene.width, scene.height = width, height
    scene.VPM[0] += (width / 2 - 640.0) * scene.VPM[3]
    scene.VPM[1] += (height / 2 - 360.0) * scene.VPM[3]
    scene.scales = scene.scales * 2.0 ** fat
    scene = scene.to(cuda)
    s = scene.settings(RasterizerMode(mode), K)
    one = FrameBuffers(*scene.gaussians(), s, True, False)
    free = FrameBuffers(*scene.gaussians(), s, True, False, waves_per_tile=waves, long_list_threshold=-1)
    image, _ = one.run()
    got, _ = free.run()
    lengths = (free.ranges[:, 1] - free.ranges[:, 0]).cpu()
    print(f"lists up to {int(lengths.max())}, chosen {int(free.long_tiles[5])}", flush=True)
    assert int(free.long_tiles[5]) == chosen(lengths, waves)
    assert (got - image).abs().max() < 3e-6
    assert torch.equal(free.run()[0], got)
