"""Lists of the tiles that a Gaussian's outline meets (``htgs_frame.touch``) against the lists of whole rectangles: no
(tile, Gaussian) pair that reaches a pixel is left out, and what is computed from the lists is the same bit for bit."""
import ctypes

import pytest
import torch

from htgs_amd import _native
from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode, rasterize, update_max_weights
from htgs_amd.torch_bindings.rasterization import run_max_weights

pytestmark = pytest.mark.gpu


def build(kind, cuda):
    g = torch.Generator().manual_seed(11)
    scene = make_scene({"near": 3, "unit": 0}.get(kind, 2), {"near": 30_000, "unit": 10_000}.get(kind, 40_000))
    n = scene.positions.shape[0]
    if kind == "needles":                      # one long axis, two of a thousandth of it
        scene.scales = torch.exp(torch.randn(n, 1, generator=g) - 3.0) * torch.tensor([[1.0, 1e-3, 1e-3]])
    elif kind == "dust":                       # far below a pixel
        scene.scales = torch.exp(torch.randn(n, 3, generator=g) - 9.0)
    elif kind == "faint":                      # opacities around the alpha thresholds
        scene.opacities = torch.exp(torch.rand(n, 1, generator=g) * 3.0) / 300.0
    elif kind == "large":                      # rectangles of far more than 64 tiles, partly outside the image
        scene.scales = torch.exp(torch.randn(n, 3, generator=g) * 0.7 - 2.0)
        scene.positions[:, :2] *= 3.0
        keep = slice(0, 3000)
        for name in ("positions", "scales", "rotations", "opacities", "sh_0", "sh_rest"):
            setattr(scene, name, getattr(scene, name)[keep].contiguous())
    return scene.to(cuda)


def pairs(fb):
    counts = torch.zeros(4, dtype=torch.int64, device=fb.device)
    _native.check(fb.lib.htgs_check_tile_cull(ctypes.byref(fb.frame), fb.selector, counts.data_ptr()))
    seen, empty, _, wrong = counts.tolist()
    assert wrong == 0
    return seen, seen - empty


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("kind", ["cluster", "near", "unit", "needles", "dust", "faint", "large"])
def test_no_pair_that_reaches_a_pixel_is_left_out(cuda, kind, mode):
    print(f"case kind={kind} mode={mode}", flush=True)
    scene = build(kind, cuda)
    s = scene.settings(RasterizerMode(mode), 16, scale_modifier=1.3 if kind == "cluster" else 1.0)
    # (the walk that keeps alphas as floats: the keys' fraction depends on the length of the list)
    whole = FrameBuffers(*scene.gaussians(), s, True, False, long_list_threshold=2 ** 30)
    tight = FrameBuffers(*scene.gaussians(), s, True, False, long_list_threshold=2 ** 30, tight_lists=True)
    image, depth = (t.clone() for t in whole.run())
    tight.run()
    assert torch.equal(tight.image, image) and torch.equal(tight.depth, depth)
    (seen, reaching), (tight_seen, tight_reaching) = pairs(whole), pairs(tight)
    assert tight_reaching == reaching and tight_seen == tight.n_instances < seen
    if kind == "cluster":
        assert tight_seen < 0.9 * seen


@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("kind", ["cluster", "near", "large"])
def test_training_and_max_weights(cuda, kind, mode):
    print(f"case kind={kind} mode={mode}", flush=True)
    scene = build(kind, cuda)
    s = scene.settings(RasterizerMode(mode), 16)
    n = scene.positions.shape[0]
    up = torch.randn(3, scene.height, scene.width, generator=torch.Generator().manual_seed(3)).to(cuda)
    results = []
    for tight in (False, True):
        fb = FrameBuffers(*scene.gaussians(), s, True, False, train=True, long_list_threshold=2 ** 30, tight_lists=tight)
        info = torch.zeros(3, n, device=cuda)
        image = fb.run_forward().clone()
        results.append((image, fb.run_backward(up, info, True), info, fb.n_instances))
    (image, grads, info, whole), (tight_image, tight_grads, tight_info, listed) = results
    assert torch.equal(image, tight_image) and listed < whole
    # (a Gaussian's rows are added up in groups that depend on their number)
    for a, b in zip((*grads, info), (*tight_grads, tight_info)):
        assert (a - b).norm() <= 1e-5 * a.norm()
    assert torch.equal(info[0], tight_info[0])
    got, want = torch.zeros(n, device=cuda), torch.zeros(n, device=cuda)
    update_max_weights(got, *scene.gaussians()[:4], s, 1e-4)
    run_max_weights(want, *scene.gaussians()[:4], s, 1e-4)
    if kind == "near":                         # (very long lists: the tail's sums are added up in parts of the list)
        assert (got - want).abs().max() < 1e-5
    else:
        assert torch.equal(got, want)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_four_byte_keys(cuda, mode):
    """More than 65536 tiles: 32-bit keys, in index order and with the Gaussians sorted by depth first."""
    scene = make_scene(0, 3000).to(cuda)
    s = scene.settings(RasterizerMode(mode), 4)._replace(width=4200, height=4200 if mode == 2 else 1100)
    image, _ = rasterize(*scene.gaussians(), s, True, False)
    want, _ = FrameBuffers(*scene.gaussians(), s, True, False).run()
    assert (image - want).abs().max() < 1e-5
