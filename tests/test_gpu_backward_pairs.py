"""The backward blend numbers the (Gaussian, quadrant) pairs of 256 instances at a time and gives a wave those of the Gaussians whose
first pair is one of 61 in a row: lists around the chunk of 256 and around a turn, with Gaussians that reach one quadrant of their
tile and Gaussians that reach all four, against the CPU oracle's gradients."""
import numpy as np
import pytest
import torch

import oracle
from htgs_amd.torch_bindings import RasterizerMode, diff_rasterize
from util import oracle_frame, tie_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [2, 3])
@pytest.mark.parametrize("mode,K", [(0, 16), (0, 32), (1, 4), (3, 1)])
@pytest.mark.parametrize("kind,n", [("wide", 1), ("wide", 15), ("wide", 16), ("narrow", 60), ("narrow", 61), ("narrow", 62), ("mixed", 245), ("mixed", 256), ("mixed", 257),
                                    ("wide", 600)])
def test_gradients_around_turns_and_chunks(cuda, kind, n, mode, K, rows):
    print(f"case kind={kind} n={n} mode={mode} K={K} rows={rows}", flush=True)
    rng = np.random.default_rng(n)
    scene = tie_scene(rng.uniform(1.0, 9.0, n).tolist(), rng.uniform(0.02, 0.9, n).tolist(), rng.uniform(0.1, 0.9, (n, 3)).tolist())
    if kind != "wide":                                       # a pixel wide, in one quadrant of the tile around pixel (36, 36)
        narrow = np.ones(n, bool) if kind == "narrow" else rng.random(n) < 0.5
        at = rng.integers(33, 39, (n, 2)) + 0.1
        z = scene.positions[:, 2].numpy()
        for axis in (0, 1):
            scene.positions[:, axis] = torch.from_numpy(np.where(narrow, (at[:, axis] - 32.0) / 100.0 * z, 0.0).astype(np.float32))
        scene.scales[torch.from_numpy(narrow)] *= 0.06
    # (an isotropic Gaussian has no gradient in its rotation but rounding)
    scene.scales *= torch.from_numpy(rng.uniform(0.6, 1.4, (n, 3)).astype(np.float32))
    scene.rotations = torch.nn.functional.normalize(torch.from_numpy(rng.standard_normal((n, 4)).astype(np.float32)))
    fr = oracle_frame(scene, mode, K)
    arrays = [t.numpy() for t in scene.gaussians()]
    fwd = oracle.forward(fr, *arrays)
    grad = rng.standard_normal((3, scene.height, scene.width)).astype(np.float32)
    want = oracle.backward(fwd, grad, *arrays)
    leaves = [t.to(cuda).requires_grad_() for t in scene.gaussians()]
    info = torch.zeros(rows, n, device=cuda)
    image = diff_rasterize(*leaves, info, scene.to(cuda).settings(RasterizerMode(mode), K), True)
    got = torch.autograd.grad(image, [t for t in leaves if t.numel()], torch.from_numpy(grad).to(cuda))
    torch.cuda.synchronize()
    assert np.abs(image.detach().cpu().numpy() - fwd["image"]).max() <= 1e-4
    names = [k for k, t in zip(("positions", "scales", "rotations", "opacities", "sh_0", "sh_rest"), leaves) if t.numel()]
    for name, g in zip(names, got):
        w = want[name].reshape(g.shape)
        assert np.abs(g.cpu().numpy() - w).max() <= 1e-3 * max(float(np.abs(w).max()), 1e-20), name
