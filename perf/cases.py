"""The work that a user of the rasterizer has it do, as a list of cases.

Every case goes through the public operators of ``htgs_amd.torch_bindings`` with tensors that are resident on the GPU,
as the renderer, the trainer and the pruning step of a splatting program call them:

* ``render``       one ``rasterize`` call: viewer frames and evaluation images (any blend mode, either image layout,
                   mean or median depth);
* ``render_fast``  one ``fast_rasterize`` call: the image alone, as a viewer or a frame-rate measurement takes it;
* ``train``        one ``diff_rasterize`` forward and its backward pass for all six Gaussian tensors, with the
                   densification statistics of none, two or three rows that the trainer asks for;
* ``max_weights``  one view of the importance-based pruning;
* ``filter_3d``    one view of the 3-D filter's update.

The Gaussians follow the distributions of the repository's own scenes (``htgs_amd/synthetic.py``): a unit cube of small
Gaussians in front of a small camera, a wide cluster in front of a 720p or 1080p camera, and a stress scene in which a
fifth of the Gaussians hug the near plane and cover much of the image.
"""
import math

import torch

from htgs_amd.synthetic import CFG3_FOCAL, SH_C0, pinhole
from htgs_amd.torch_bindings import (RasterizerMode, RasterizerSettings, diff_rasterize, fast_rasterize, rasterize,
                                     update_3d_filter, update_max_weights)

HYBRID, FIRST_K, GLOBAL, OIT = 0, 1, 2, 3
NEAR, FAR = 0.2, 1000.0
CLUSTER_DISTANCE = 12.0


def _case(name, op, n, width, height, mode=HYBRID, K=16, scene="cluster", log_scale=-4.5, sh_total=16, sh_active=16, chw=True, median=False, rows=0):
    return {"name": name, "op": op, "n": n, "width": width, "height": height, "mode": mode, "K": K, "scene": scene, "log_scale": log_scale,
            "sh_total": sh_total, "sh_active": sh_active, "chw": chw, "median": median, "rows": rows}


def listed():
    return [
        # a thumbnail of a small object: every launch and every line of host code counts
        _case("render-tiny-256", "render", 10_000, 256, 256, K=4, scene="unit", log_scale=-4.0, sh_total=1, sh_active=1),
        # an ordinary viewer frame without the order-independent tail
        _case("render-720p-first-k", "render", 1_000_000, 1280, 720, mode=FIRST_K),
        # the frame that the framework's headline figure is quoted on: the default mode and core size, full HD
        _case("render-1080p-hybrid", "render", 3_000_000, 1920, 1080),
        # the same scene with globally sorted alpha blending, what other splatting programs do
        _case("render-1080p-global", "render", 3_000_000, 1920, 1080, mode=GLOBAL),
        # an evaluation image of a dataset whose photographs have an odd size, channels last, median depth
        _case("render-odd-oit-median", "render", 333_667, 1237, 821, mode=OIT, chw=False, median=True),
        # a camera inside the scene: Gaussians at the near plane cover much of the image, lists of 100 000 and more
        _case("render-stress-6M", "render", 6_000_000, 1600, 1066, scene="stress", log_scale=-3.0),
        # the image alone, as fast as it can be had
        _case("render-fast-1080p", "render_fast", 3_000_000, 1920, 1080),
        # an early training step: few Gaussians, a downscaled image, the higher SH bands not yet active
        _case("train-early-small", "train", 20_000, 400, 304, log_scale=-3.5, sh_active=1, rows=2),
        # a training step in the middle of a run with two rows of densification statistics
        _case("train-1080p-hybrid", "train", 1_000_000, 1920, 1080, rows=2),
        # a training step of the globally sorted mode on an odd image size, with the third row (absolute gradients)
        _case("train-odd-global", "train", 411_111, 1297, 839, mode=GLOBAL, rows=3),
        # one view of importance-based pruning, which goes over all training views
        _case("max-weights-1080p", "max_weights", 1_000_000, 1920, 1080),
        # one view of the 3-D filter's update, which also goes over all training views
        _case("filter-3d-3M", "filter_3d", 3_000_000, 1920, 1080),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: any operator, any mode, 10 thousand to 6 million Gaussians, images of 256 to 1920
    by 256 to 1080 pixels, any core size and SH degree; never more work than the stress frame or the large training step."""
    while True:
        op = rng.choice(["render"] * 4 + ["train"] * 4 + ["render_fast", "max_weights", "filter_3d"])
        n = _log_uniform(rng, 10_000, 1_000_000 if op == "train" else 3_000_000)
        scene = "stress" if op != "filter_3d" and rng.random() < 0.15 else "cluster"
        if scene == "stress":
            n = min(n, 600_000 if op in ("train", "max_weights") else 3_000_000)
        width, height = _log_uniform(rng, 256, 1920), _log_uniform(rng, 256, 1080)
        sh_total = rng.choice([1, 4, 9, 16, 16, 16])
        sh_active = rng.choice([b for b in (1, 4, 9, 16) if b <= sh_total] + [sh_total])
        # the fewer Gaussians a scene has, the larger they are
        log_scale = -3.0 if scene == "stress" else round(-4.5 + math.log(1e6 / n) / 3.0 * rng.uniform(0.0, 1.0), 3)
        case = _case("", op, n, width, height, mode=rng.randrange(4), K=rng.choice([4, 8, 16, 16, 16, 32]), scene=scene, log_scale=log_scale,
                     sh_total=sh_total, sh_active=sh_active, chw=rng.random() < 0.7, median=rng.random() < 0.3,
                     rows=rng.choice([0, 2, 3]) if op == "train" else 0)
        del case["name"]
        most = 4e8 if op in ("train", "max_weights") else 2e9
        if _fragments(case) <= most:
            return case


def _focal(case):
    """Pixels.  The repository's cameras: 1.17 (the small scene) and 0.78 (the clusters) of the image's width."""
    return {"unit": case["width"] * 300.0 / 256.0, "cluster": case["width"] * 0.78125, "stress": CFG3_FOCAL * case["width"] / 1600.0}[case["scene"]]


def _scale_sigma(case):
    return {"unit": 0.5, "cluster": 0.7, "stress": 0.8}[case["scene"]]


def _gaussians(case, g, dev):
    n = case["n"]

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    def rand(*shape):
        return torch.rand(*shape, generator=g, device=dev)

    if case["scene"] == "unit":
        positions = rand(n, 3) * 2.0 - 1.0
        positions[:, 2] += 4.0
    elif case["scene"] == "cluster":
        positions = randn(n, 3) * 2.0
        positions *= torch.clamp(10.0 / positions.norm(dim=1, keepdim=True).clamp_min(1e-12), max=1.0)
    else:
        d = randn(n, 3)
        positions = d / d.norm(dim=1, keepdim=True).clamp_min(1e-12) * (6.0 * rand(n, 1) ** (1.0 / 3.0))
        positions[:, 2] += 4.0
        near = rand(n, 1) < 0.2
        hugging = torch.cat([(rand(n, 2) * 2.0 - 1.0) * 0.5, 0.2 + 0.5 * rand(n, 1)], dim=1)
        positions = torch.where(near, hugging, positions).contiguous()
    scales = torch.exp(randn(n, 3) * _scale_sigma(case) + case["log_scale"])
    rotations = randn(n, 4)
    rotations /= rotations.norm(dim=1, keepdim=True).clamp_min(1e-12)
    opacities = torch.sigmoid(randn(n, 1) * (1.0 if case["scene"] == "unit" else 1.5))
    sh_0 = (rand(n, 1, 3) - 0.5) / SH_C0
    sh_rest = randn(n, case["sh_total"] - 1, 3) * 0.05
    return positions, scales, rotations, opacities, sh_0, sh_rest


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    width, height, f = case["width"], case["height"], _focal(case)
    M, VPM, cam_position = pinhole(width, height, f, f, width / 2, height / 2, NEAR, FAR,
                                   translation=(0.0, 0.0, CLUSTER_DISTANCE if case["scene"] == "cluster" else 0.0))
    settings = RasterizerSettings(M.to(dev), VPM.to(dev), cam_position.to(dev), RasterizerMode(case["mode"]), case["K"], case["sh_active"], width, height,
                                  NEAR, FAR, 1.0)
    state = {"case": case, "settings": settings}
    if case["op"] == "filter_3d":
        state["gaussians"] = (_gaussians(dict(case, sh_total=1), g, dev)[0],)
        state["filter"] = torch.full((case["n"], 1), 1.0e9, device=dev)
        state["visible"] = torch.zeros(case["n"], dtype=torch.bool, device=dev)
        return state
    state["gaussians"] = _gaussians(case, g, dev)
    if case["op"] == "train":
        state["gaussians"] = tuple(t.requires_grad_() for t in state["gaussians"])
        state["grad_image"] = torch.randn(3, height, width, generator=g, device=dev)
        state["densification_info"] = torch.zeros((case["rows"], case["n"]) if case["rows"] else (0,), device=dev)
    elif case["op"] == "max_weights":
        state["max_weights"] = torch.zeros(case["n"], device=dev)
    return state


def run(state):
    case, settings, gaussians = state["case"], state["settings"], state["gaussians"]
    op = case["op"]
    if op == "render":
        return rasterize(*gaussians, settings, case["chw"], case["median"])
    if op == "render_fast":
        return fast_rasterize(*gaussians, settings, case["chw"])
    if op == "train":
        info = state["densification_info"]
        image = diff_rasterize(*gaussians, info, settings, case["rows"] > 0)
        grads = torch.autograd.grad(image, gaussians, state["grad_image"])
        return [image.detach(), *grads, info]
    if op == "max_weights":
        update_max_weights(state["max_weights"], *gaussians[:4], settings, 0.02)
        return state["max_weights"]
    f = _focal(case)
    update_3d_filter(*gaussians, settings.M, state["filter"], state["visible"], case["width"], case["height"], f, f, case["width"] / 2.0,
                     case["height"] / 2.0, NEAR, 0.15, math.sqrt(0.2) / f)
    return [state["filter"], state["visible"]]


def _fragments(case):
    """(pixel, Gaussian) pairs inside the Gaussians' cut-off ellipses, from the distributions: a randomly turned ellipsoid
    with half axes s1, s2, s3 (times the cut-off radius) projects to about pi E[s_i s_j] (f / z)^2 pixels, at most the
    image; E[s_i s_j] = exp(2 mu + sigma^2) for independent log-normal axes.  The squared radius is 2 ln(255 opacity)
    (2 ln(20 opacity) where the least alpha is 1/20), about 9.4 (4.6) on average over the opacities; what falls beyond
    the image's edge is not taken off."""
    radius_sq = 4.6 if case["mode"] == FIRST_K else 9.4
    area = math.pi * radius_sq * math.exp(2.0 * case["log_scale"] + _scale_sigma(case) ** 2) * _focal(case) ** 2
    image = float(case["width"] * case["height"])
    if case["scene"] == "unit":
        per_gaussian = area / 15.0                        # E[1 / z^2] for z in [3, 5]
    elif case["scene"] == "cluster":
        per_gaussian = area * 1.09 / CLUSTER_DISTANCE ** 2
    else:
        # a fifth at z in [0.2, 0.7] (E[1 / z^2] = 1 / 0.14), the others around z = 4, of which four fifths are in front
        per_gaussian = 0.2 * min(area / 0.14, 0.25 * image) + 0.64 * min(area / 10.0, 0.25 * image)
    return case["n"] * min(per_gaussian, image)


# operations that a fragment costs: two planes, the point nearest to the Gaussian, the exponential and the blend; the
# backward pass evaluates it again and takes the gradient through the same steps
FORWARD_FLOPS, BACKWARD_FLOPS = 70, 210


def work(case):
    n, pixels, B = case["n"], case["width"] * case["height"], case["sh_active"]
    op = case["op"]
    if op == "filter_3d":
        return {"bytes": n * (12 + 4 + 4 + 1), "flops": 24 * n}
    geometry = 4 * (3 + 3 + 4 + 1)
    if op == "max_weights":
        return {"bytes": n * (geometry + 8), "flops": FORWARD_FLOPS * _fragments(case)}
    read = n * (geometry + 12 * B)
    if op == "train":
        # the six gradients (the inactive bands' zeros among them), the upstream gradient, the statistics
        return {"bytes": read + n * (geometry + 12 * case["sh_total"] + 8 * case["rows"]) + 24 * pixels,
                "flops": (FORWARD_FLOPS + BACKWARD_FLOPS) * _fragments(case)}
    return {"bytes": read + (12 if op == "render_fast" else 16) * pixels, "flops": FORWARD_FLOPS * _fragments(case)}


def tolerance(case):
    """Sums of 32-bit products in another order: 1e-5 in images, depths and weights, ten times that in gradients, whose terms
    cancel.  A fragment within rounding of an alpha threshold moves a single pixel by up to a twentieth (a gradient
    entry by its share), which the largest difference allows for; the fast path takes the hardware's reciprocal and power
    of two, so more of its fragments do."""
    op = case["op"]
    if op == "filter_3d":
        return {"rel": 1e-6}
    if op == "train":
        return {"rel": 1e-4, "max": 0.05}
    if op == "render_fast":
        return {"rel": 1e-4, "max": 0.2}
    return {"rel": 2e-5, "max": 0.05}
