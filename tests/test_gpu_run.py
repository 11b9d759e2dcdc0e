"""Whole passes by ``htgs_run``: a frame that is queued before the host knows its number of instances equals the frame taken
stage by stage, whether the number comes out as expected, larger (queued a second time), smaller or zero."""
import ctypes
import threading
import types
from typing import NamedTuple

import pytest
import torch

from htgs_amd import _native
from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode, diff_rasterize, fast_rasterize, rasterize, update_max_weights
from htgs_amd.torch_bindings.rasterization import ScratchPool, current_stream_handle, run_max_weights

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


@pytest.mark.parametrize("op,mode,K,lines", [("render", 0, 16, {6144: 4, 15360: 2}), ("render", 1, 4, {6144: 4, 15360: 2}), ("render", 0, 32, {6144: 4, 13312: 2}),
                                             ("render", 3, 1, {6144: 4, 16384: 2}), ("render_fast", 0, 16, {6144: 4, 13312: 2}), ("render", 2, 1, {}),
                                             ("train", 0, 16, {6144: 4, 10240: 2}), ("train", 1, 4, {6144: 4, 10240: 2}), ("train", 1, 32, {6144: 4, 8192: 2}),
                                             ("train", 0, 32, {8192: 2}), ("train", 3, 1, {6144: 4, 16384: 2}), ("max_weights", 0, 16, {})])
def test_waves_per_tile_on_both_sides_of_the_lines(cuda, op, mode, K, lines):
    """At the lines' own grids and one column of tiles beyond, the number of waves, and the result against one wave a tile."""
    pool = ScratchPool.current(cuda)
    for rows, beside in ((48, 128), (64, 128), (80, 128), (104, 128), (120, 128), (128, 128)):
        for columns in (beside, beside + 1):
            scene = make_scene(1, 3000)
            scene.width, scene.height = 8 * columns, 8 * rows
            scene = scene.to(cuda)
            s = scene.settings(RasterizerMode(mode), K)
            tiles = rows * columns
            want = next((w for line, w in lines.items() if tiles <= line), 1)
            print(f"case {op} mode={mode} K={K} tiles={tiles} waves={want}", flush=True)
            if op == "train":
                leaves = [t.clone().requires_grad_() for t in scene.gaussians()]
                image = diff_rasterize(*leaves, torch.empty(0, device=cuda), s, False)
                assert image.grad_fn.fb.frame.waves_per_tile == want
                one = FrameBuffers(*scene.gaussians(), s, True, False, train=True).run_forward()
            elif op == "max_weights":
                weights = torch.zeros(3000, device=cuda)
                update_max_weights(weights, *scene.gaussians()[:4], s, 0.01)
                assert pool.frame.waves_per_tile == want
                continue
            else:
                image = fast_rasterize(*scene.gaussians(), s, True) if op == "render_fast" else rasterize(*scene.gaussians(), s, True, False)[0]
                assert pool.frame.waves_per_tile == want
                one = FrameBuffers(*scene.gaussians(), s, True, False, fast=op == "render_fast").run()[0]
            assert (image.detach() - one).abs().max() < 3e-6


class Reordered(NamedTuple):
    note: str
    scale_modifier: float
    far_plane: float
    near_plane: float
    height: int
    width: int
    K: int
    mode: RasterizerMode
    active_sh_bases: int
    VPM: torch.Tensor
    cam_position: torch.Tensor
    M: torch.Tensor


class Fresh:
    """An object whose matrices are new tensors each time they are read."""
    def __init__(self, s):
        self.s = s

    def __getattr__(self, name):
        v = getattr(self.s, name)
        return v.clone() if isinstance(v, torch.Tensor) else v


@pytest.mark.parametrize("kind", ["namespace", "reordered", "fresh"])
def test_settings_are_any_object_with_the_attributes(cuda, kind):
    scene = make_scene(0, 3000).to(cuda)
    s = scene.settings(RasterizerMode.HYBRID_BLEND, 4, scale_modifier=1.2)
    other = {"namespace": lambda: types.SimpleNamespace(**s._asdict()), "reordered": lambda: Reordered(note="", **s._asdict()), "fresh": lambda: Fresh(s)}[kind]()
    print(f"case {kind}", flush=True)
    for a, b in zip(rasterize(*scene.gaussians(), s, True, False), rasterize(*scene.gaussians(), other, True, False)):
        assert torch.equal(a, b)
    assert torch.equal(fast_rasterize(*scene.gaussians(), s, True), fast_rasterize(*scene.gaussians(), other, True))
    results = []
    for settings in (s, other):
        leaves = [t.clone().requires_grad_() for t in scene.gaussians()]
        image = diff_rasterize(*leaves, torch.empty(0, device=cuda), settings, False)
        if kind == "namespace":                              # (what the forward pass was given is what the backward pass uses)
            kept, other.M, other.VPM, other.cam_position = (other.M, other.VPM, other.cam_position), None, None, None
        junk = [torch.full((4, 4), 7.0, device=cuda) for _ in range(8)]
        results.append((image.detach(), *torch.autograd.grad(image, leaves, torch.ones_like(image))))
        del junk
        if kind == "namespace":
            other.M, other.VPM, other.cam_position = kept
        weights = torch.zeros(3000, device=cuda)
        update_max_weights(weights, *scene.gaussians()[:4], settings, 0.01)
        results[-1] += (weights,)
    for a, b in zip(*results):
        assert torch.equal(a, b)


def views(scene, cuda):
    """The scene from farther and nearer, up and down: instances between one and two and a half times the least."""
    for distance in (0.0, -1.3, 0.4, -1.6, -0.8, 1.0, -1.6, -1.9):
        M, VPM = scene.M.clone(), scene.VPM.clone()
        M[:, 3] += distance * torch.tensor([0.0, 0.0, 1.0, 0.0])
        VPM[:, 3] += distance * scene.VPM[:, 2]
        yield scene.settings(RasterizerMode.HYBRID_BLEND, 4)._replace(M=M.to(cuda), VPM=VPM.to(cuda), cam_position=torch.tensor([0.0, 0.0, -distance], device=cuda))


@pytest.mark.parametrize("n,mode", [(3000, 0), (3000, 2), (80_000, 0), (80_000, 1), (80_000, 2), (80_000, 3)])
def test_changing_views(cuda, n, mode):
    """More instances than the buffers hold or the launches were sized for, with the blend queued ahead (3000 Gaussians) and behind the
    number (80 000), with the scan in the duplication and, where the Gaussians are sorted by depth first, on its own: images, gradients and weights of a sequence of views against the stages; a training frame
    keeps the workspace that it was rendered with and no other."""
    scene = make_scene(0, n)
    todo, scene_gpu = [s._replace(mode=RasterizerMode(mode)) for s in views(scene, cuda)], scene.to(cuda)
    g = scene_gpu.gaussians()
    up = torch.randn(3, scene.height, scene.width, generator=torch.Generator().manual_seed(4)).to(cuda)
    def same(a, b, at_most):                                 # (long lists are walked in shares, whose sums come in another order)
        assert torch.equal(a, b) if n == 3000 else (a - b).abs().max() < at_most
    ScratchPool.clear()
    counts, again = [], 0
    for i, s in enumerate(todo):
        print(f"case n={n} mode={mode} view={i}", flush=True)
        expected = ScratchPool.current(cuda).expected((1, mode))
        image, depth = rasterize(*g, s, True, False)
        want, want_depth = FrameBuffers(*g, s, True, False, tight_lists=True, waves_per_tile=4).run()
        same(image, want, 3e-6)
        same(depth[0], want_depth, 5e-5)
        leaves = [t.clone().requires_grad_() for t in g]
        image = diff_rasterize(*leaves, torch.empty(0, device=cuda), s, False)
        frame = image.grad_fn.fb
        assert sum(t.dtype == torch.uint8 for t in frame.keep if isinstance(t, torch.Tensor)) == 2
        counts.append(frame.frame.n_instances)
        again += expected != 0 and counts[-1] > expected + expected // 8 + 4096
        fb = FrameBuffers(*g, s, True, False, train=True, tight_lists=True, waves_per_tile=4)
        same(image.detach(), fb.run_forward(), 3e-6)
        for a, b in zip(torch.autograd.grad(image, leaves, up), fb.run_backward(up)):
            assert (a - b).norm() <= (0.0 if n == 3000 else 1e-4) * b.norm()
        got, ref = torch.zeros(n, device=cuda), torch.zeros(n, device=cuda)
        update_max_weights(got, *g[:4], s, 0.01)
        run_max_weights(ref, *g[:4], s, 0.01)
        assert (got - ref).abs().max() < 1e-5                # (the tail's sums in shares of the list)
    assert max(counts) > 1.5 * min(counts) and again >= (1 if n > 3000 else 0)


def test_transposed_camera_matrices_take_the_same_path(cuda):
    scene = make_scene(0, 3000).to(cuda)
    s = scene.settings(RasterizerMode.HYBRID_BLEND, 4)
    views_of = s._replace(M=s.M.t().contiguous().t(), VPM=s.VPM.t().contiguous().t(), cam_position=torch.stack([s.cam_position] * 2, 1)[:, 0])
    assert not (views_of.M.is_contiguous() or views_of.VPM.is_contiguous() or views_of.cam_position.is_contiguous())
    assert torch.equal(rasterize(*scene.gaussians(), views_of, True, False)[0], rasterize(*scene.gaussians(), s, True, False)[0])
    results = []
    for settings in (s, views_of):
        leaves = [t.clone().requires_grad_() for t in scene.gaussians()]
        image = diff_rasterize(*leaves, torch.empty(0, device=cuda), settings, False)
        assert image.grad_fn.fb.fallback is None
        results.append((image.detach(), *torch.autograd.grad(image, leaves, torch.ones_like(image))))
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_threads_and_streams(cuda):
    """Four threads, each on a stream of its own, with views that change from call to call: every image and every gradient is that of
    the pass on its own."""
    scene = make_scene(0, 70_000)
    todo, scene_gpu = list(views(scene, cuda)), scene.to(cuda)
    g = scene_gpu.gaussians()
    def one(k, i):
        s = todo[(3 * k + i) % len(todo)]._replace(mode=RasterizerMode((k + i) % 4))
        image, _ = rasterize(*g, s, True, False)
        leaves = [t.detach().clone().requires_grad_() for t in g]
        trained = diff_rasterize(*leaves, torch.empty(0, device=cuda), s, False)
        return [image, trained.detach(), *torch.autograd.grad(trained, leaves, torch.ones_like(trained))]
    want = [[one(k, i) for i in range(6)] for k in range(4)]
    torch.cuda.synchronize()
    failures = []
    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for i in range(6):
                    got = one(k, i)
                    torch.cuda.current_stream().synchronize()
                    if not all(torch.equal(a, b) for a, b in zip(got, want[k][i])):
                        failures.append((k, i))
                torch.cuda.current_stream().synchronize()
        except Exception as e:                               # (shown by the assertion below)
            failures.append((k, repr(e)))
    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


@pytest.mark.parametrize("most", [3, 86])
def test_scan_of_more_sums_than_every_block_adds_up(cuda, most):
    """49152 blocks of 2048 counts and two more, the last one short: offsets against torch's, and the total (86: beyond 2^32 - 2)."""
    n = 49152 * 2048 + 2048 + 77
    print(f"case n={n} most={most}", flush=True)
    f = _native.Frame()
    counts = torch.randint(0, most + 1, (n,), dtype=torch.int32, device=cuda, generator=torch.Generator(device=cuda).manual_seed(7))
    offsets, total = torch.empty(n, dtype=torch.int32, device=cuda), torch.empty(1, dtype=torch.int32, device=cuda)
    tmp = torch.empty(_native.lib().htgs_scan_tmp_words(n), dtype=torch.int32, device=cuda)
    f.n_primitives, f.width, f.height, f.mode = n, 64, 64, 0
    f.n_touched, f.offsets, f.scan_tmp, f.n_instances_dev = counts.data_ptr(), offsets.data_ptr(), tmp.data_ptr(), total.data_ptr()
    f.stream = torch.cuda.current_stream().cuda_stream
    _native.check(_native.lib().htgs_scan_offsets(ctypes.byref(f)))
    want = torch.cumsum(counts, 0, dtype=torch.int64)
    assert (int(total) & 0xffffffff) == (int(want[-1]) if most == 3 else 0xffffffff)
    assert torch.equal(offsets, want.to(torch.int32))        # (modulo 2^32 where the frame is refused)


def test_pass_with_more_block_sums_than_every_block_adds_up(cuda):
    """12.6 M Gaussians, 256 to a sum: the image of the pass against the stages, whose sums are of 2048."""
    n = 49152 * 256 + 3 * 256 + 19
    print(f"case n={n}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(5)
    scene = make_scene(0, 1000).to(cuda)
    positions = torch.rand(n, 3, generator=g, device=cuda) * 2.0 - 1.0
    positions[:, 2] += torch.where(torch.rand(n, generator=g, device=cuda) < 0.02, 4.0, -400.0)        # (most of them behind the camera)
    gaussians = (positions, torch.full((n, 3), 4e-3, device=cuda), torch.tensor([[1.0, 0.0, 0.0, 0.0]], device=cuda).repeat(n, 1),
                 torch.full((n, 1), 0.3, device=cuda), torch.randn(n, 1, 3, generator=g, device=cuda), torch.zeros(n, 0, 3, device=cuda))
    s = scene.settings(RasterizerMode.OIT_BLEND, 1)
    want, _ = FrameBuffers(*gaussians, s, True, False, tight_lists=True, waves_per_tile=4).run()
    for _ in range(2):                                       # (the number of instances unknown, then expected)
        image, _ = rasterize(*gaussians, s, True, False)
        assert (image - want).abs().max() < 3e-6 and float(image.mean()) > 0.05


@pytest.mark.parametrize("mode,fast", [(0, False), (1, False), (2, False), (3, False), (0, True)])
def test_stages_like_a_pass(cuda, mode, fast):
    """``FrameBuffers.like`` has the lists that the pass had: as many instances, the same image."""
    scene = make_scene(1, 60_000).to(cuda)
    s = scene.settings(RasterizerMode(mode), 16)
    image = fast_rasterize(*scene.gaussians(), s, True) if fast else rasterize(*scene.gaussians(), s, True, False)[0]
    frame = ScratchPool.current(cuda).frame
    n, waves = frame.n_instances, frame.waves_per_tile
    fb = FrameBuffers.like(frame, *scene.gaussians(), s, True, False, fast=fast)
    assert torch.equal(fb.run()[0], image) and fb.n_instances == n and fb.frame.waves_per_tile == waves


def test_current_stream_handle(cuda):
    """The stream that a pass is queued on: torch's current one, of the device asked for, with or without an index."""
    for device in (cuda, torch.device("cuda")):
        assert current_stream_handle(device) == torch.cuda.current_stream(device).cuda_stream
        side = torch.cuda.Stream(device)
        with torch.cuda.stream(side):
            assert current_stream_handle(device) == side.cuda_stream != 0
        assert current_stream_handle(device) == torch.cuda.current_stream(device).cuda_stream


@pytest.mark.parametrize("parameters", [False, True])
def test_gradients_are_plain_contiguous_tensors(cuda, parameters):
    """Gradients laid out as documented whatever the inputs are: parameters, tensors, views with odd strides of dimensions of one."""
    scene = make_scene(1, 300).to(cuda)
    given = [t.requires_grad_() for t in scene.gaussians()]
    if parameters:
        given = [torch.nn.Parameter(t.detach()) for t in given]
    else:
        given[3] = torch.as_strided(given[3].detach(), (300, 1), (1, 7)).requires_grad_()
        given[4] = torch.as_strided(given[4].detach(), (300, 1, 3), (3, 11, 1)).requires_grad_()
    image = diff_rasterize(*given, torch.empty(0, device=cuda), scene.settings(RasterizerMode(0), 4), False)
    for t, grad in zip(given, torch.autograd.grad(image, given, torch.ones_like(image))):
        assert type(grad) is torch.Tensor and grad.shape == t.shape and grad.is_contiguous() and not grad.requires_grad
