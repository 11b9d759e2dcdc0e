"""Instances made bin by bin of depth (``htgs_frame.depth_bins``) against lists by Gaussian index: the lists themselves, and what the
walks make of them where fragments of exactly equal depth meet, whose order by index the reference's insertion depends on
(R/include/hybrid_blend/kernels/inference.cuh:159-167)."""
import dataclasses

import pytest
import torch

from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode, diff_rasterize, fast_rasterize, rasterize, update_max_weights
from htgs_amd.torch_bindings.rasterization import ScratchPool, run_max_weights
from test_gpu_long_tiles import with_coincident_copies

pytestmark = pytest.mark.gpu

HYBRID, FIRST_K = 0, 1


def small_view(scene, width=203, height=149):
    scene.VPM[0] += (width / 2 - scene.width / 2) * scene.VPM[3]
    scene.VPM[1] += (height / 2 - scene.height / 2) * scene.VPM[3]
    scene.width, scene.height = width, height
    return scene


def with_twins(scene, twins):
    """The first ``twins`` Gaussians once more, among the others by index, with other colours and opacities: pairs of fragments of
    exactly equal depth wherever they are."""
    n = scene.positions.shape[0]
    order = torch.cat([torch.arange(n), torch.arange(twins)])[torch.randperm(n + twins, generator=torch.Generator().manual_seed(5))]
    pick = lambda t: t[order].contiguous()
    g = torch.Generator().manual_seed(6)
    return dataclasses.replace(
        scene, positions=pick(scene.positions), scales=pick(scene.scales), rotations=pick(scene.rotations), sh_rest=pick(scene.sh_rest),
        opacities=(pick(scene.opacities) * (0.6 + 0.4 * torch.rand(n + twins, 1, generator=g))).contiguous(),
        sh_0=(pick(scene.sh_0) + 0.5 * torch.randn(n + twins, *scene.sh_0.shape[1:], generator=g)).contiguous())


def build(kind):
    if kind == "twins":
        return with_twins(small_view(make_scene(1, 40_000)), 20_000)
    if kind == "copies":
        return with_coincident_copies(make_scene(0, 1500), 4)
    return make_scene(3, 60_000) if kind == "near" else small_view(make_scene(1, 60_000), 640, 400)


def frame(sg, mode, K, bins, **kwargs):
    return FrameBuffers(*sg.gaussians(), sg.settings(RasterizerMode(mode), K), True, kwargs.pop("median", False), tight_lists=True, depth_bins=bins, long_counters=True, **kwargs)


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("n", [1, 63, 257, 70_001])
def test_lists(cuda, n, train):
    """Every tile's list holds the same Gaussians as without bins, in up to eight runs by index, of growing depth; a training frame's
    offsets say where each Gaussian's instances are."""
    sg = small_view(make_scene(1, n), 640, 400).to(cuda)
    by_index, binned = (frame(sg, HYBRID, 16, bins, train=train) for bins in (False, True))
    for fb in (by_index, binned):
        fb.preprocess()
        fb.scan()
        fb.alloc_instances(fb.read_instance_count())
        fb.create_instances()
    m = by_index.n_instances
    assert binned.n_instances == m and torch.equal(binned.n_touched, by_index.n_touched)
    unsorted = binned.vals[0][:m].clone()
    for fb in (by_index, binned):
        fb.selector = fb.sort()
        fb.extract_ranges()
    assert torch.equal(binned.ranges, by_index.ranges)
    pairs = [torch.stack([fb.keys[fb.selector][:m].to(torch.int64), fb.vals[fb.selector][:m].to(torch.int64)]) for fb in (by_index, binned)]
    assert torch.equal(pairs[0][:, torch.argsort(pairs[0][0] * n + pairs[0][1])], pairs[1][:, torch.argsort(pairs[1][0] * n + pairs[1][1])])
    if m > 1:
        same_tile = pairs[1][0][1:] == pairs[1][0][:-1]
        back = same_tile & (pairs[1][1][1:] < pairs[1][1][:-1])
        assert int(torch.bincount(pairs[1][0][1:][back], minlength=1).max()) <= 7
        # a run ends where a nearer bin's depths end: behind a step back by index nothing is nearer than what came before the step's run
        z = (sg.positions.to(torch.float64) @ sg.M.to(torch.float64)[2, :3] + sg.M.to(torch.float64)[2, 3])[unsorted.to(torch.int64)]
        steps = torch.nonzero(unsorted[1:] < unsorted[:-1]).flatten() + 1
        assert len(steps) <= 7
        for step in steps.tolist():
            assert float(z[:step].max()) <= float(z[step:].min()) + 1e-5
    if train:
        ends, counts = binned.offsets.to(torch.int64), binned.n_touched.to(torch.int64)
        seen = torch.nonzero(counts).flatten()
        slots = torch.repeat_interleave(ends[seen] - counts[seen], counts[seen]) + torch.cat([torch.arange(int(c), device=cuda) for c in counts[seen].tolist()] or [counts[:0]])
        assert torch.equal(unsorted[slots].to(torch.int64), torch.repeat_interleave(seen, counts[seen]))


@pytest.mark.parametrize("n,scans", [(1, 2), (257, 2), (70_001, 3), (4_194_304, 1), (4_194_305, 1), (4_300_001, 2)])
def test_scan(cuda, n, scans):
    """The scan of the bins may be called again, and takes more than one round of 4 194 304 Gaussians: as many instances as by index, each in
    the same tile."""
    print(f"case n={n} scans={scans}", flush=True)
    sg = small_view(make_scene(1, min(n, 70_001)), 640, 400).to(cuda)
    if n > 70_001:
        more = lambda t: t.repeat(n // 70_001 + 1, *[1] * (t.ndim - 1))[:n].contiguous()
        g = torch.Generator(device=cuda).manual_seed(1)
        sg = dataclasses.replace(sg, positions=more(sg.positions) + 0.05 * torch.randn(n, 3, generator=g, device=cuda), scales=more(sg.scales), rotations=more(sg.rotations),
                                 opacities=more(sg.opacities), sh_0=more(sg.sh_0), sh_rest=torch.zeros(n, 0, 3, device=cuda), active_sh_bases=1)
    pairs = []
    for bins in (False, True):
        fb = frame(sg, HYBRID, 16, bins)
        fb.preprocess()
        for _ in range(scans):
            fb.scan()
        fb.alloc_instances(fb.read_instance_count())
        fb.create_instances()
        m = fb.n_instances
        pairs.append(torch.sort((fb.keys[0][:m].to(torch.int64) & 0xffff) * n + fb.vals[0][:m].to(torch.int64)).values)
    assert torch.equal(*pairs)


@pytest.mark.parametrize("waves,threshold", [(1, 0), (2, 0), (4, 0), (1, 60)])
@pytest.mark.parametrize("K", [1, 2, 4, 16, 32])
@pytest.mark.parametrize("mode", [HYBRID, FIRST_K])
@pytest.mark.parametrize("kind", ["twins", "copies", "near", "plain"])
def test_image_and_depth(cuda, kind, mode, K, waves, threshold):
    """Pairs of equal depth inside a core and at its end, more than two of a depth, near-plane scenes, chance ties: the walk by insertion over
    the list by index (threshold above 8192) is what both orders have to come to.  Bounds: the keys' rounding of alpha (2^-20 at most)
    and the tail's sums in another order, as for the walks by index."""
    print(f"case kind={kind} mode={mode} K={K} waves={waves} threshold={threshold}", flush=True)
    sg = build(kind).to(cuda)
    want, want_depth = frame(sg, mode, K, False, long_list_threshold=2 ** 31 - 1).run()
    got, got_depth = frame(sg, mode, K, True, waves_per_tile=waves, long_list_threshold=threshold).run()
    assert (got - want).abs().max() < 4e-6
    assert (got_depth - want_depth).abs().max() < 1e-4


@pytest.mark.parametrize("waves,threshold", [(1, 0), (2, 0), (1, 60)])
@pytest.mark.parametrize("K", [1, 4, 16, 32])
@pytest.mark.parametrize("mode", [HYBRID, FIRST_K])
@pytest.mark.parametrize("kind", ["twins", "copies", "plain"])
def test_training(cuda, kind, mode, K, waves, threshold):
    """The same core indices, slot by slot; gradients of the rows wherever they are."""
    print(f"case kind={kind} mode={mode} K={K} waves={waves} threshold={threshold}", flush=True)
    sg = build(kind).to(cuda)
    frames = [frame(sg, mode, K, bins, train=True, waves_per_tile=waves if bins else 1, long_list_threshold=threshold if bins else 2 ** 31 - 1) for bins in (False, True)]
    images = [fb.run_forward() for fb in frames]
    assert (images[1] - images[0]).abs().max() < 4e-6
    assert torch.equal(*[fb.records_in_image_order(fb.core_idx) for fb in frames])
    grad_image = torch.randn(images[0].shape, generator=torch.Generator(device=cuda).manual_seed(3), device=cuda)
    for a, b in zip(*[fb.run_backward(grad_image, None, False) for fb in frames]):
        assert a.numel() == 0 or (a - b).abs().max() <= 1e-4 * max(1e-6, float(a.abs().max()))


@pytest.mark.parametrize("mode", [HYBRID, FIRST_K])
def test_operators(cuda, mode):
    """340 000 Gaussians, a third of them twins, on a grid of one wave a tile: the operators take bins, and come to what the stages by index come to."""
    print(f"case mode={mode}", flush=True)
    sg = with_twins(small_view(make_scene(1, 240_000), 1300, 1000), 100_000).to(cuda)
    s = sg.settings(RasterizerMode(mode), 16)
    image, depth = rasterize(*sg.gaussians(), s, True, False)
    assert ScratchPool.current(cuda).frame.depth_bins
    want, want_depth = frame(sg, mode, 16, False, long_list_threshold=2 ** 31 - 1).run()
    assert (image - want).abs().max() < 4e-6 and (depth[0] - want_depth).abs().max() < 1e-4
    step = diff_rasterize(*[t.requires_grad_() for t in sg.gaussians()], torch.empty(0, device=cuda), s, False)
    assert step.grad_fn.fb.frame.depth_bins
    by_index = frame(sg, mode, 16, False, train=True, long_list_threshold=2 ** 31 - 1)
    assert (step.detach() - by_index.run_forward()).abs().max() < 4e-6
    weights, by_stages = torch.zeros(340_000, device=cuda), torch.zeros(340_000, device=cuda)
    with torch.no_grad():
        update_max_weights(weights, *[t.detach() for t in sg.gaussians()[:4]], s, 0.02)
        run_max_weights(by_stages, *[t.detach() for t in sg.gaussians()[:4]], s, 0.02, long_list_threshold=2 ** 31 - 1)
    if mode == FIRST_K:
        assert torch.equal(weights, by_stages)
    else:
        # (a weight within rounding of the threshold may fall on the other side of it)
        both = (weights > 0) & (by_stages > 0)
        assert ((weights - by_stages).abs()[both] <= 1e-5 * by_stages[both]).all() and int((both != ((weights > 0) | (by_stages > 0))).sum()) <= 2


def within_fast_bounds(fast, exact):
    """What the image-only path may differ by (tests/test_gpu_parity.py): a fragment within an ulp of an alpha threshold is decided differently,
    1/20 of a colour at most, in fewer than a pixel of a thousand."""
    diff = (fast - exact).abs()
    return float((diff > 1e-5).float().mean()) < 1e-3 and float(diff.max()) <= 5e-2


@pytest.mark.parametrize("waves,threshold", [(1, 0), (2, 0), (4, 0), (1, 60)])
@pytest.mark.parametrize("K", [1, 8, 16, 32])
@pytest.mark.parametrize("mode", [HYBRID, FIRST_K])
@pytest.mark.parametrize("kind", ["plain", "near"])
def test_image_alone(cuda, kind, mode, K, waves, threshold):
    """The image-only kernels over lists in bins, against the exact walk by insertion over the list by index."""
    print(f"case kind={kind} mode={mode} K={K} waves={waves} threshold={threshold}", flush=True)
    sg = build(kind).to(cuda)
    want, _ = frame(sg, mode, K, False, long_list_threshold=2 ** 31 - 1).run()
    fb = frame(sg, mode, K, True, fast=True, order_gaussians=False, waves_per_tile=waves, long_list_threshold=threshold)
    got, _ = fb.run()
    assert fb.frame.depth_bins and not fb.frame.depth_order
    assert within_fast_bounds(got, want)


@pytest.mark.parametrize("K", [8, 16, 32])
@pytest.mark.parametrize("mode", [HYBRID, FIRST_K])
def test_fast_operator(cuda, mode, K):
    """``fast_rasterize`` takes bins for 810 000 Gaussians on a grid of one wave a tile."""
    print(f"case mode={mode} K={K}", flush=True)
    sg = small_view(make_scene(1, 810_000), 1300, 1000).to(cuda)
    s = sg.settings(RasterizerMode(mode), K)
    got = fast_rasterize(*sg.gaussians(), s, True)
    assert ScratchPool.current(cuda).frame.depth_bins
    assert within_fast_bounds(got, frame(sg, mode, K, False, long_list_threshold=2 ** 31 - 1).run()[0])


@pytest.mark.parametrize("width,height,n,bins", [(640, 480, 340_000, False), (1300, 1000, 199_999, False), (1300, 1000, 340_000, True)])
def test_lines(cuda, width, height, n, bins):
    """Grids that four waves share a tile of take no bins at these sizes; what the operators return does not depend on it."""
    sg = small_view(make_scene(1, n), width, height).to(cuda)
    s = sg.settings(RasterizerMode(HYBRID), 16)
    image, depth = rasterize(*sg.gaussians(), s, True, False)
    assert bool(ScratchPool.current(cuda).frame.depth_bins) == bins
    want, want_depth = frame(sg, HYBRID, 16, False, long_list_threshold=2 ** 31 - 1).run()
    assert (image - want).abs().max() < 4e-6 and (depth[0] - want_depth).abs().max() < 1e-4
