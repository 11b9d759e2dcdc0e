"""The backward blend numbers the (Gaussian, quadrant) pairs of 256 instances at a time and gives a wave those of the Gaussians whose
first pair is one of 61 in a row: lists around the chunk of 256 and around a turn, with Gaussians that reach one quadrant of their
tile and Gaussians that reach all four, against the CPU oracle's gradients and densification statistics.  The rows of a Gaussian are
added up four at a time by four lanes up to sixteen rows and by the whole wave beyond: exact sums of whole numbers."""
import numpy as np
import pytest
import torch

import oracle
from htgs_amd.synthetic import make_scene
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode, diff_rasterize
from util import oracle_frame, tie_scene, u32

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
    want_info = np.zeros((rows, n), np.float32)
    want = oracle.backward(fwd, grad, *arrays, densification_info=want_info, use_distance_scaling=True)
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
    got_info = info.cpu().numpy()
    np.testing.assert_array_equal(got_info[0], want_info[0])
    for r in range(1, rows):                                 # (norms and sums of the gradients' size, none of them cancel)
        assert np.abs(got_info[r] - want_info[r]).max() <= 1e-3 * max(float(want_info[r].max()), 1e-20), r
    assert rows == 2 or want_info[2].max() > 0.0


@pytest.mark.parametrize("n", [1, 63, 64, 255, 257, 2000])
def test_rows_of_a_gaussian_are_added_up(cuda, n):
    """Rows of whole numbers, whose sums are exact in any order: the gradients are those of one row with the sum and rows of zeros."""
    print(f"case n={n}", flush=True)
    scene = make_scene(0, n)
    scene.width, scene.height = 203, 149
    scene.VPM[0] += (scene.width / 2 - 128.0) * scene.VPM[3]
    scene.VPM[1] += (scene.height / 2 - 128.0) * scene.VPM[3]
    g = torch.Generator().manual_seed(n)
    if n > 1:
        scene.scales *= torch.exp(torch.rand(n, 1, generator=g) * 2.5)
    gpu = scene.to(cuda)
    fb = FrameBuffers(*gpu.gaussians(), gpu.settings(RasterizerMode.HYBRID_BLEND, 4), True, False, train=True, tight_lists=True)
    fb.run_forward()
    info = torch.zeros(3, n, device=cuda)
    fb.run_backward(torch.ones(3, scene.height, scene.width, device=cuda), info)
    helper = fb._backward_buffers[2]
    counts, ends = u32(fb.n_touched).astype(np.int64), u32(fb.offsets).astype(np.int64)
    assert n < 2000 or set(range(22)) <= set(counts.tolist())
    rows = torch.randint(-1000, 1001, (fb.n_instances, 16), generator=g).float()
    helped = torch.randint(0, 1001, (fb.n_instances,), generator=g).float()
    sums, total = torch.zeros_like(rows), torch.zeros_like(helped)
    for i in np.flatnonzero(counts):
        sums[ends[i] - counts[i]] = rows[ends[i] - counts[i]:ends[i]].sum(0)
        total[ends[i] - counts[i]] = helped[ends[i] - counts[i]:ends[i]].sum()
    results = []
    for r, h in ((rows, helped), (sums, total)):
        fb.grad_rows[:fb.n_instances] = r.to(cuda)
        helper[:fb.n_instances] = h.to(cuda)
        info.zero_()
        fb.preprocess_backward()
        results.append([t.clone() for t in (*fb.grads, info)])
    for a, b in zip(*results):
        assert torch.equal(a, b)
    drawn = torch.from_numpy(counts > 0)
    start = torch.from_numpy(ends - counts)[drawn]
    assert torch.equal(results[0][3].reshape(-1).cpu()[drawn], sums[start, 3]) and torch.equal(results[0][6][2].cpu()[drawn], total[start])


@pytest.mark.parametrize("K", [1, 2, 8, 16, 32])
@pytest.mark.parametrize("kind,times,more", [("wide", 4, -1), ("wide", 4, 0), ("mixed", 8, 0), ("wide", 0, 256), ("mixed", 0, 257), ("wide", 0, 770)])
def test_gradients_of_core_members(cuda, kind, times, more, K):
    """ALPHA_BLEND_FIRST_K leaves out what is in no core of a quadrant, in lists from 4 K on, a chunk of 256 at a time."""
    for rows in (2, 3):
        test_gradients_around_turns_and_chunks(cuda, kind, times * K + more, 1, K, rows)


@pytest.mark.parametrize("rows", [2, 3])
@pytest.mark.parametrize("kind,n", [("wide", 1), ("wide", 26), ("wide", 27), ("wide", 28), ("narrow", 63), ("narrow", 64), ("narrow", 65), ("mixed", 130), ("mixed", 400), ("wide", 200)])
def test_gradients_around_batches_of_pairs(cuda, kind, n, rows):
    """ALPHA_BLEND_GLOBAL_ORDERING takes 64 Gaussians at a time, or as many as have 432 (Gaussian, quadrant) pairs: 27 that reach all sixteen."""
    test_gradients_around_turns_and_chunks(cuda, kind, n, 2, 1, rows)
