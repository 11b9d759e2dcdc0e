"""The duplication of masks goes through a window of 2048 instances in LDS, masks of up to twelve tiles lane by lane and larger ones by the
whole wave, or up to twenty-four lane by lane in a wave with more than twelve masks between the two: blocks of 256 Gaussians with few and
many instances, masks around twelve tiles, around twenty-four and the largest, against the instances listed one rectangle at a time on the host."""
import numpy as np
import pytest
import torch

from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode
from util import tie_scene, u32

pytestmark = pytest.mark.gpu


def listed(fb):
    """Per Gaussian the tiles of its touch entry, from the entry itself."""
    touch = u32(fb.touch).reshape(-1, 4)
    counts = u32(fb.n_touched)
    pairs = []
    for g in np.flatnonzero(counts):
        corner, size, lo, hi = (int(v) for v in touch[g])
        x0, y0, w, h = corner & 0xffff, corner >> 16, size & 0xffff, size >> 16
        if w * h > 64:
            return None
        mask = lo | hi << 32
        tiles = [(y0 + b // w) * fb.grid_w + x0 + b % w for b in range(64) if mask >> b & 1]
        assert len(tiles) == counts[g]
        pairs += [(t, g) for t in tiles]
    return sorted(pairs)


@pytest.mark.parametrize("mode", [0, 2, 3])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 700])
@pytest.mark.parametrize("spread", ["small", "around twelve", "around twenty-four", "few large", "largest"])
def test_instances_of_masks(cuda, spread, n, mode):
    print(f"case spread={spread} n={n} mode={mode}", flush=True)
    rng = np.random.default_rng(n)
    scene = tie_scene(rng.uniform(1.0, 9.0, n).tolist(), rng.uniform(0.3, 1.0, n).tolist(), rng.uniform(0.0, 1.0, (n, 3)).tolist())
    scene.scales *= {"small": 0.2, "around twelve": 1.0, "around twenty-four": 1.4, "few large": 0.3, "largest": 2.0}[spread] * torch.from_numpy(rng.uniform(0.6, 1.0, (n, 1)).astype(np.float32))
    scene.positions[:, :2] = torch.from_numpy(rng.uniform(-0.2, 0.2, (n, 2)).astype(np.float32)) * scene.positions[:, 2:3]
    if spread == "few large":
        scene.scales[torch.from_numpy(rng.random(n) < 0.12)] *= 5.0
    gpu = scene.to(cuda)
    fb = FrameBuffers(*gpu.gaussians(), gpu.settings(RasterizerMode(mode), 4), True, False, tight_lists=True, order_gaussians=False)
    fb.preprocess()
    fb.scan()
    count = fb.read_instance_count()
    fb.alloc_instances(count)
    fb.create_instances()
    torch.cuda.synchronize()
    want = listed(fb)
    assert want is not None and len(want) == count            # (an 8x8 grid: every rectangle has a mask)
    if mode != 2 and n >= 255 and spread not in ("small", "largest"):
        sizes = np.pad(u32(fb.n_touched), (0, -n % 64)).reshape(-1, 64)
        between, beyond = ((sizes > 12) & (sizes <= 24)).sum(1), (sizes > 24).sum(1)
        print("between:", between.tolist(), "beyond:", beyond.tolist())
        if spread == "few large":                            # the line at twelve, and masks on both sides of it
            assert between.max() <= 12 and between.any() and beyond.any()
        else:                                                # the line at twenty-four
            assert between.max() > 12 and (beyond.any() or spread == "around twelve")
    keys = u32(fb.keys[0])[:count].astype(np.uint64)
    tiles = keys >> np.uint64(32) if mode == 2 else keys
    got = list(zip(tiles.astype(np.int64).tolist(), u32(fb.vals[0])[:count].tolist()))
    assert [g for _, g in got] == sorted(g for _, g in got)   # in the Gaussians' order, which the stable sort keeps
    assert sorted(got) == want


@pytest.mark.parametrize("mode", [0, 2, 3])
@pytest.mark.parametrize("by", [256, 1024])
def test_instances_on_a_grid_beyond_two_to_the_twenty_tiles(cuda, by, mode):
    """The duplication on its own, with offsets from elsewhere (the scan stops at 2^20 tiles): an entry of the window counts its tile from
    the mask's corner, whose number has 32 bits.  (Grids of 2^21 and 2^25 tiles; the stages in question have no image and no ranges.)"""
    print(f"case by={by} mode={mode}", flush=True)
    n = 1000
    rng = np.random.default_rng(3)
    scene = tie_scene(rng.uniform(1.0, 9.0, n).tolist(), rng.uniform(0.3, 1.0, n).tolist(), rng.uniform(0.0, 1.0, (n, 3)).tolist())
    scene.positions[:, :2] = torch.from_numpy(rng.uniform(-0.3, 0.3, (n, 2)).astype(np.float32)) * scene.positions[:, 2:3]
    by *= 2 if mode == 2 else 1                              # (tiles of twice the edge)
    scene.VPM[0] *= by
    scene.VPM[1] *= by / 2.0
    scene.scales *= 1.0 / by
    gpu = scene.to(cuda)
    fb = FrameBuffers(*gpu.gaussians(), gpu.settings(RasterizerMode(mode), 4), True, False, tight_lists=True, order_gaussians=False)
    fb.frame.width, fb.frame.height = 64 * by + 16, 32 * by + 16
    fb.grid_w = (fb.frame.width + fb.tile - 1) // fb.tile
    fb.key_bytes = fb.lib.htgs_frame_key_bytes(fb._ref)
    assert fb.key_bytes == (8 if mode == 2 else 4)
    fb.preprocess()
    offsets = torch.cumsum(fb.n_touched, 0).to(torch.int32)
    fb.offsets.copy_(offsets)
    count = int(offsets[-1])
    fb.alloc_instances(count)
    fb.create_instances()
    torch.cuda.synchronize()
    want = listed(fb)
    assert want is not None and len(want) == count
    assert max(t for t, _ in want) > (1 << 20 if by <= 512 else 1 << 24)
    keys = u32(fb.keys[0])[:count].astype(np.uint64)
    tiles = keys >> np.uint64(32) if mode == 2 else keys
    assert sorted(zip(tiles.astype(np.int64).tolist(), u32(fb.vals[0])[:count].tolist())) == want
