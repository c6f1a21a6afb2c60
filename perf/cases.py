"""Performance cases: the work a user of this framework has it do.

A case is one call sequence of a training or viewing program: rendering a
model, a training step (render, image loss, gradients of every parameter), or
one of the operators a program composes by itself. Sizes and distributions are
those of ``gsplat_core.scenes`` and of the benchmark (10,000 Gaussians at
256x256 up to 6,000,000 at 3840x2160, or 8 cameras at once), made on the GPU
from the seed. ``exact`` restates each path in plain float64 torch.
"""
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "gsplat-mlx_amd"))

import gsplat_core as G  # noqa: E402
from gsplat_core import render as R  # noqa: E402

TILE = 16
SSIM_WINDOW = 11  # the trainer's defaults: window 11, (1 - 0.2) L1 + 0.2 (1 - SSIM) / 2
SSIM_LAMBDA = 0.2

# What a scene's Gaussians look like: centre and spread of the means, of the
# log-scales and of the opacity logits, the focal length per image width, the
# background and the far plane.
#   box    a unit box of flat-coloured Gaussians in front of the camera
#   panel  a wide slab of flat-coloured Gaussians, fitted to one image
#   seed   a capture's point cloud before training: few, large, faint Gaussians
#   cloud  a trained capture: a million small Gaussians around the view axis
#   ring   the same centred at the origin, cameras on a ring around it
#   dense  a far, wide scene at high resolution with long tile lists
SCENES = {
    "box": {"focal": 1.0, "far": 1e10, "bg": 0.0},
    "panel": {"focal": 1.0, "far": 1e10, "bg": 0.0},
    "seed": {"focal": 1150.0 / 1297.0, "far": 100.0, "bg": 0.025},
    "cloud": {"focal": 1150.0 / 1297.0, "far": 100.0, "bg": 0.025},
    "ring": {"focal": 1600.0 / 1920.0, "far": 100.0, "bg": 0.025},
    "dense": {"focal": 3000.0 / 3840.0, "far": 100.0, "bg": 0.025},
}

# (pixel, Gaussian) pairs that contribute to the image, per pixel: in
# proportion to the Gaussians until the pixels saturate (measured: pairs per
# pixel and Gaussian of a sparse scene, pairs per pixel of a full one).
PAIRS = {"box": (2.6e-3, 73.0), "panel": (1.0e-3, 73.0), "seed": (1.1e-3, 136.0), "cloud": (3.0e-4, 73.0),
         "ring": (2.0e-4, 73.0), "dense": (2.0e-4, 65.0)}


def listed():
    return [
        # a preview of a small model: launches and the count read-back matter
        {"name": "view_box_10k", "kind": "view_rgb", "scene": "box", "n": 10_000, "width": 256, "height": 256,
         "cameras": 1, "accutile": False},
        # one iteration of fitting flat-coloured Gaussians to an image
        {"name": "fit_panel_100k", "kind": "fit_rgb", "scene": "panel", "n": 100_000, "width": 512, "height": 512,
         "cameras": 1, "accutile": False},
        # the first thousands of iterations of a capture's training: the point
        # cloud, SH degree 1 of 3, L1 + DSSIM
        {"name": "train_seed_120k", "kind": "train_sh", "scene": "seed", "n": 120_000, "width": 1297, "height": 840,
         "cameras": 1, "degree": 1, "loss": "l1_dssim", "accutile": False, "packed": False},
        # a viewer's frame of a trained capture
        {"name": "view_cloud_1m", "kind": "view_sh", "scene": "cloud", "n": 1_000_000, "width": 1297, "height": 840,
         "cameras": 1, "degree": 3, "accutile": False, "packed": False},
        # the benchmark's training step
        {"name": "train_cloud_1m", "kind": "train_sh", "scene": "cloud", "n": 1_000_000, "width": 1297, "height": 840,
         "cameras": 1, "degree": 3, "loss": "l1", "accutile": False, "packed": False},
        # ellipse tile lists and the trainer's default loss, odd sizes
        {"name": "train_ellipse_713k", "kind": "train_sh", "scene": "cloud", "n": 713_117, "width": 1237,
         "height": 822, "cameras": 1, "degree": 3, "loss": "l1_dssim", "accutile": True, "packed": False},
        # the packed layout over several cameras
        {"name": "train_packed_500k", "kind": "train_sh", "scene": "ring", "n": 500_009, "width": 979, "height": 545,
         "cameras": 4, "degree": 3, "loss": "l1", "accutile": False, "packed": True},
        # a batch of 8 full-HD cameras over 3M Gaussians
        {"name": "train_ring_3m", "kind": "train_sh", "scene": "ring", "n": 3_000_000, "width": 1920, "height": 1080,
         "cameras": 8, "degree": 3, "loss": "l1", "accutile": False, "packed": False},
        # 6M Gaussians at 4K: a quarter of a billion tile entries
        {"name": "train_dense_6m", "kind": "train_sh", "scene": "dense", "n": 6_000_000, "width": 3840,
         "height": 2160, "cameras": 1, "degree": 3, "loss": "l1", "accutile": False, "packed": False},
        # the projection operator both ways with compensations, two cameras
        {"name": "project_800k", "kind": "project", "scene": "ring", "n": 800_003, "width": 1297, "height": 840,
         "cameras": 2, "model": 0, "compensations": True},
        # the spherical harmonics operator both ways with direction gradients
        {"name": "harmonics_600k", "kind": "harmonics", "n": 600_011, "degree": 3},
        # the sorted tile lists and their offsets for two images
        {"name": "lists_200k", "kind": "lists", "scene": "cloud", "n": 200_001, "width": 1001, "height": 667,
         "cameras": 2},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["view_rgb", "fit_rgb", "view_sh", "train_sh", "train_sh", "train_sh", "train_dense", "train_ring",
                       "project", "harmonics", "lists"])
    width = _log_uniform(rng, 160, 1600)
    height = max(96, int(width * rng.uniform(0.5, 1.0)))
    case = {"kind": kind, "n": _log_uniform(rng, 5_000, 1_000_000), "width": width, "height": height, "cameras": 1}
    options = {"accutile": rng.random() < 0.25, "packed": rng.random() < 0.25}
    if kind in ("view_rgb", "fit_rgb"):
        return dict(case, scene=rng.choice(["box", "panel"]), n=_log_uniform(rng, 1_000, 200_000),
                    width=min(width, 800), height=min(height, 800), cameras=rng.choice([1, 1, 2]),
                    accutile=options["accutile"])
    if kind == "view_sh":
        return dict(case, scene="cloud", degree=rng.choice([0, 1, 2, 3, 3]), **options)
    if kind == "train_sh":
        scene = rng.choice(["seed", "cloud", "cloud"])
        if scene == "seed":
            case["n"] = _log_uniform(rng, 5_000, 200_000)
        return dict(case, scene=scene, degree=rng.choice([0, 1, 2, 3, 3]), loss=rng.choice(["l1", "l1_dssim"]),
                    **options)
    if kind == "train_dense":
        width = _log_uniform(rng, 1024, 3840)
        return dict(case, kind="train_sh", scene="dense", n=_log_uniform(rng, 300_000, 6_000_000), width=width,
                    height=width * 9 // 16, degree=3, loss="l1", accutile=False, packed=False)
    if kind == "train_ring":
        return dict(case, kind="train_sh", scene="ring", n=_log_uniform(rng, 100_000, 1_500_000),
                    cameras=rng.randint(2, 8), degree=3, loss=rng.choice(["l1", "l1_dssim"]), **options)
    if kind == "project":
        return dict(case, scene="ring", n=_log_uniform(rng, 20_000, 2_000_000), cameras=rng.randint(1, 4),
                    model=rng.choice([0, 0, 1, 2]), compensations=rng.random() < 0.5)
    if kind == "harmonics":
        return {"kind": kind, "n": _log_uniform(rng, 20_000, 2_000_000), "degree": rng.randint(0, 4)}
    return dict(case, scene="cloud", cameras=rng.randint(1, 4))


# --------------------------------------------------------------------- inputs


def _views(scene, cameras, dtype=torch.float32):
    """World-to-camera matrices [1, C, 4, 4]: a ring of radius 8 looking at the
    origin, or cameras a little beside each other looking along z."""
    views = np.tile(np.eye(4), (1, cameras, 1, 1))
    for c in range(cameras):
        if scene == "ring":
            a = 2 * math.pi * c / max(cameras, 3)
            rot = np.array([[math.cos(a), 0, math.sin(a)], [0, 1, 0], [-math.sin(a), 0, math.cos(a)]])
            views[0, c, :3, :3] = rot
            views[0, c, 2, 3] = 8.0
        else:
            views[0, c, 0, 3] = 0.1 * c
    return torch.from_numpy(views.astype(np.float32)).to(dtype)


def _intrinsics(case):
    f = SCENES[case["scene"]]["focal"] * case["width"]
    K = torch.tensor([[f, 0, case["width"] / 2], [0, f, case["height"] / 2], [0, 0, 1]], dtype=torch.float32)
    return K.expand(1, case["cameras"], 3, 3).contiguous()


def _gaussians(case, gen):
    n, scene, dev = case["n"], case["scene"], "cuda"

    def normal(shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=gen, device=dev) * std + mean

    def uniform(shape, low, high):
        return torch.rand(shape, generator=gen, device=dev) * (high - low) + low

    if scene in ("box", "panel"):
        half, near, far = (1.0, 3.0, 5.0) if scene == "box" else (2.0, 3.0, 6.0)
        means = torch.cat([uniform((1, n, 2), -half, half), uniform((1, n, 1), near, far)], -1)
        return {"means": means, "quats": normal((1, n, 4)), "log_scales": uniform((1, n, 3), -5.0, -2.0),
                "opacity_logits": normal((1, n)), "colors": uniform((1, n, 3), 0.0, 1.0)}
    means, scales, logits = normal((1, n, 3)), normal((1, n, 3)), normal((1, n))
    if scene == "dense":
        means = means * torch.tensor([7.0, 3.94, 6.0], device=dev) + torch.tensor([0.0, 0.0, 30.0], device=dev)
        scales = scales * 0.7 - 2.5
        logits = torch.where(uniform((1, n), 0.0, 1.0) < 0.3, logits + 3.0, logits - 1.0)
    else:
        means = means * 2.0
        if scene != "ring":
            means[..., 2] += 6.0
        scales = scales * 0.5 - (3.2 if scene == "seed" else 4.0)
        if scene == "seed":
            logits = logits * 0.3 - 2.0
    rest = {"means": means, "quats": normal((1, n, 4)), "log_scales": scales, "opacity_logits": logits}
    if "degree" in case:
        rest["features_dc"] = normal((1, n, 3), 0.0, 0.3)
        rest["features_rest"] = normal((1, n, 15, 3), 0.0, 0.05)
    return rest


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, n = case["kind"], case["n"]
    if kind == "harmonics":
        K = (case["degree"] + 1) ** 2
        return {"case": case,
                "dirs": torch.randn((n, 3), generator=gen, device="cuda").requires_grad_(True),
                "coeffs": (torch.randn((n, K, 3), generator=gen, device="cuda") * 0.2).requires_grad_(True),
                "v_colors": torch.randn((n, 3), generator=gen, device="cuda")}
    C, W, H = case["cameras"], case["width"], case["height"]
    if kind == "lists":
        # projected Gaussians: centres over and around the image, radii of a
        # few pixels with some large ones, a fifth unseen. The seed gives their
        # order and depths, so every seed's lists have the same length.
        fixed = torch.Generator(device="cuda").manual_seed(n)
        centre = torch.rand((1, C, n, 2), generator=fixed, device="cuda") * 1.1 - 0.05
        radii = torch.exp(torch.randn((1, C, n, 2), generator=fixed, device="cuda") * 0.9 + 1.6).ceil().int()
        radii[:, :, : n // 5] = 0
        order = torch.randperm(n, generator=gen, device="cuda")
        return {"case": case,
                "inputs": {"means2d": (centre * torch.tensor([float(W), float(H)], device="cuda"))[:, :, order],
                           "radii": radii[:, :, order],
                           "depths": torch.rand((1, C, n), generator=gen, device="cuda") * 12.0 + 0.2}}
    state = {"case": case, "viewmats": _views(case["scene"], C).cuda(), "Ks": _intrinsics(case).cuda(),
             "params": _gaussians(case, gen)}
    if kind == "project":
        p = state["params"]
        p["quats"] = p["quats"] / p["quats"].norm(dim=-1, keepdim=True)
        p["scales"] = torch.exp(p.pop("log_scales"))
        p.pop("opacity_logits")
        shape = (1, C, n)
        state["cotangents"] = [torch.randn(shape + (k,) if k else shape, generator=gen, device="cuda")
                               for k in (2, 0, 3, 0)]
    if kind in ("fit_rgb", "train_sh"):
        state["target"] = torch.rand((C, H, W, 3), generator=gen, device="cuda")
        state["one"] = torch.ones((), device="cuda")
    if kind in ("train_sh", "project"):
        for p in state["params"].values():
            p.requires_grad_(True)
    if kind == "train_sh":
        state["viewspace"] = torch.zeros((1, C, n, 2), device="cuda", requires_grad=True)
    return state


# ----------------------------------------------------------------------- runs


def _render_sh(state, viewspace=None):
    case, p = state["case"], state["params"]
    scene = SCENES[case["scene"]]
    return R.render_sh_model(p["means"], p["quats"], p["log_scales"], p["features_dc"], p["features_rest"],
                             p["opacity_logits"], state["viewmats"], state["Ks"], case["width"], case["height"], TILE,
                             case["degree"], viewspace_points=viewspace, background=(scene["bg"],) * 3,
                             far_plane=scene["far"], accutile=case["accutile"], packed=case["packed"])


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "view_rgb":
        p = state["params"]
        with torch.no_grad():
            out = R.render_rgb_model(p["means"], p["quats"], p["log_scales"], p["colors"], p["opacity_logits"],
                                     state["viewmats"], state["Ks"], case["width"], case["height"], TILE,
                                     opacities_in_projection=True, accutile=case["accutile"])
        return [out["render_colors"], out["render_alphas"]]
    if kind == "fit_rgb":
        p = state["params"]
        loss, out, grads = R.render_rgb_model_l1_value_and_grad(
            p["means"], p["quats"], p["log_scales"], p["colors"], p["opacity_logits"], state["viewmats"], state["Ks"],
            state["target"], case["width"], case["height"], TILE, accutile=case["accutile"])
        return [loss, out["render_colors"], out["render_alphas"], grads["v_means"], grads["v_quats"],
                grads["v_log_scales"], grads["v_opacity_logits"], grads["v_colors"]]
    if kind == "view_sh":
        with torch.no_grad():
            out = _render_sh(state)
        return [out["render_colors"], out["render_alphas"]]
    if kind == "train_sh":
        leaves = list(state["params"].values()) + [state["viewspace"]]
        for leaf in leaves:
            leaf.grad = None
        out = _render_sh(state, state["viewspace"])
        if case["loss"] == "l1":
            loss = R.l1_loss(out["render_colors"], state["target"])
        else:
            loss = R.image_training_loss(out["render_colors"], state["target"], case["loss"], SSIM_LAMBDA, SSIM_WINDOW)
        loss.backward(state["one"])
        return [loss.detach(), out["render_colors"].detach(), out["render_alphas"].detach()] + [p.grad for p in leaves]
    if kind == "project":
        p = state["params"]
        for leaf in p.values():
            leaf.grad = None
        out = G.projection_ewa_3dgs_fused(p["means"], state["viewmats"], state["Ks"], case["width"], case["height"],
                                          quats=p["quats"], scales=p["scales"], far_plane=100.0,
                                          calc_compensations=case["compensations"], camera_model=case["model"])
        names = ["means2d", "depths", "conics"] + (["compensations"] if case["compensations"] else [])
        torch.autograd.backward([out[k] for k in names], state["cotangents"][: len(names)])
        return [out["radii"]] + [out[k].detach() for k in names] + [p[k].grad for k in ("means", "quats", "scales")]
    if kind == "harmonics":
        state["dirs"].grad = state["coeffs"].grad = None
        colors = G.spherical_harmonics(case["degree"], state["dirs"], state["coeffs"])
        colors.backward(state["v_colors"])
        return [colors.detach(), state["dirs"].grad, state["coeffs"].grad]
    tw, th = R.tile_grid(case["width"], case["height"], TILE)
    out = G.intersect_tile_offsets_forward(state["inputs"], case["cameras"], TILE, tw, th)
    return [out["tiles_per_gauss"], out["isect_ids"], out["flatten_ids"], out["tile_offsets"]]


# --------------------------------------------------------- work and tolerance


def work(case):
    """Each input read once, each output written once; the flops of the
    rasterizer's contributing (pixel, Gaussian) pairs (27 forward, 75
    backward) and of the per-Gaussian operators (a few hundred)."""
    n, kind = case["n"], case["kind"]
    if kind == "harmonics":
        K = (case["degree"] + 1) ** 2
        return {"bytes": n * (12 + 12 * K + 24 + 12 + 12 * K), "flops": n * K * 30}
    C, pixels = case["cameras"], case["cameras"] * case["width"] * case["height"]
    if kind == "lists":
        # a handful of tiles per seen Gaussian
        entries = int(3.3 * C * n)
        return {"bytes": C * n * 24 + entries * 12, "flops": 0}
    if kind == "project":
        rows = C * n
        per_row = 8 + 8 + 4 + 12 + (4 if case["compensations"] else 0)
        return {"bytes": n * 40 + rows * per_row + rows * (per_row - 8) + n * 80, "flops": rows * 900}
    per_gaussian, full = PAIRS[case["scene"]]
    pairs = pixels * min(per_gaussian * n, full)
    image = pixels * 16
    if kind == "view_rgb":
        return {"bytes": n * 60 + image, "flops": int(27 * pairs + 400 * n * C)}
    if kind == "fit_rgb":
        return {"bytes": n * 120 + image + pixels * 12, "flops": int(102 * pairs + 1300 * n * C)}
    coefficients = 12 * (case["degree"] + 1) ** 2
    if kind == "view_sh":
        return {"bytes": n * (48 + coefficients) + image, "flops": int(27 * pairs + 500 * n * C)}
    # the step's gradients cover all 16 coefficients
    return {"bytes": n * (44 + coefficients + 44 + 192) + C * n * 8 + image + pixels * 12,
            "flops": int(102 * pairs + 1600 * n * C)}


def tolerance(case):
    """About four times the largest distance from ``exact`` that was seen."""
    kind = case["kind"]
    if kind == "lists":
        return "exact"
    if kind in ("view_rgb", "view_sh"):
        # a pixel whose alpha or transmittance meets its threshold to the last
        # bit gains or loses a contribution of up to 1/255 (3e-5 seen in small
        # images, 2e-6 in large ones)
        return {"rel": 1.2e-4}
    if kind in ("fit_rgb", "train_sh"):
        # the same ties, and the L1 term's sign where image and target agree to
        # the last bits: one pixel's whole cotangent (2.6e-3 seen)
        return {"rel": 1e-2}
    if kind == "project":
        # a radius whose ceiling meets a whole number may differ by one
        return {"rel": 4e-5, "differ": 1e-5}
    return {"rel": 1e-6}


# ------------------------------------------------------------ float64 restated


def _rotation(q):
    w, x, y, z = q.unbind(-1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).reshape(*q.shape[:-1], 3, 3)


def _project64(case, means, quats, scales, views, Ks, far, opacities=None, model=0):
    """Projection of [n] Gaussians into C cameras: a dict of [C, n, ...]."""
    W, H = case["width"], case["height"]
    rot = _rotation(quats / quats.norm(dim=-1, keepdim=True)) if quats is not None else None
    M = rot * scales[..., None, :]
    world = M @ M.transpose(-1, -2)
    out = {k: [] for k in ("means2d", "depths", "conics", "compensations", "radii")}
    for c in range(views.shape[0]):
        V, K = views[c], Ks[c]
        fx, fy, cx, cy = K[0, 0], K[1, 1], K[0, 2], K[1, 2]
        cam = means @ V[:3, :3].T + V[:3, 3]
        cov = V[:3, :3] @ world @ V[:3, :3].T
        x, y, z = cam.unbind(-1)
        seen = (z >= 0.01) & (z <= far)
        if model != 1:
            z = torch.where(seen, z, torch.ones_like(z))
        zero = torch.zeros_like(z)
        if model == 0:
            tan_x, tan_y = 0.5 * W / fx, 0.5 * H / fy
            tx = z * (x / z).clamp(-(cx / fx + 0.3 * tan_x), (W - cx) / fx + 0.3 * tan_x)
            ty = z * (y / z).clamp(-(cy / fy + 0.3 * tan_y), (H - cy) / fy + 0.3 * tan_y)
            J = torch.stack([fx / z, zero, -fx * tx / z**2, zero, fy / z, -fy * ty / z**2], -1)
            m2 = torch.stack([fx * x / z + cx, fy * y / z + cy], -1)
        elif model == 1:
            J = torch.stack([fx + zero, zero, zero, zero, fy + zero, zero], -1)
            m2 = torch.stack([fx * x + cx, fy * y + cy], -1)
        else:
            eps = 1e-7
            r = torch.sqrt(x * x + y * y) + eps
            theta = torch.atan2(r, z + eps)
            m2 = torch.stack([x * fx * theta / r + cx, y * fy * theta / r + cy], -1)
            x2, y2, xy = x * x + eps, y * y, x * y
            b = torch.atan2(r, z) / r / (x2 + y2)
            inv = 1 / (x2 + y2 + z * z)
            a = z * inv / (x2 + y2)
            J = torch.stack([fx * (x2 * a + y2 * b), fx * xy * (a - b), -fx * x * inv,
                             fy * xy * (a - b), fy * (y2 * a + x2 * b), -fy * y * inv], -1)
        J = J.reshape(-1, 2, 3)
        cov2 = J @ cov @ J.transpose(-1, -2)
        det0 = cov2[:, 0, 0] * cov2[:, 1, 1] - cov2[:, 0, 1] * cov2[:, 1, 0]
        A, B, D = cov2[:, 0, 0] + 0.3, cov2[:, 0, 1], cov2[:, 1, 1] + 0.3
        det = A * D - B * B
        seen = seen & (det > 0)
        comp = torch.sqrt(torch.clamp(det0 / det, min=0.005**2))
        extend = torch.full_like(det, 3.33)
        if opacities is not None:
            seen = seen & (opacities >= 1 / 255)
            extend = torch.minimum(extend, torch.sqrt(2 * torch.log((opacities * 255).clamp(min=1.0))))
        with torch.no_grad():
            rx, ry = torch.ceil(extend * torch.sqrt(A)), torch.ceil(extend * torch.sqrt(D))
            seen = seen & ~((rx <= 0) & (ry <= 0))
            seen = seen & ~((m2[:, 0] + rx <= 0) | (m2[:, 0] - rx >= W) | (m2[:, 1] + ry <= 0) | (m2[:, 1] - ry >= H))
        keep = seen[:, None]
        out["means2d"].append(torch.where(keep, m2, torch.zeros_like(m2)))
        out["depths"].append(torch.where(seen, z, zero))
        conic = torch.stack([D / det, -B / det, A / det], -1)
        out["conics"].append(torch.where(keep, conic, torch.zeros_like(conic)))
        out["compensations"].append(torch.where(seen, comp, zero))
        out["radii"].append(torch.where(keep, torch.stack([rx, ry], -1), torch.zeros_like(m2.detach())).int())
    return {k: torch.stack(v) for k, v in out.items()}


def _harmonics64(degree, dirs, coeffs):
    """Real spherical harmonics (Condon-Shortley signs) of unit vectors."""
    d = dirs / dirs.norm(dim=-1, keepdim=True)
    x, y, z = d.unbind(-1)
    pi = math.pi
    basis = [torch.full_like(x, 0.5 / math.sqrt(pi))]
    if degree > 0:
        k = math.sqrt(3 / (4 * pi))
        basis += [-k * y, k * z, -k * x]
    if degree > 1:
        k = 0.5 * math.sqrt(15 / pi)
        basis += [k * x * y, -k * y * z, 0.25 * math.sqrt(5 / pi) * (3 * z * z - 1), -k * x * z,
                  0.5 * k * (x * x - y * y)]
    if degree > 2:
        a, b, c = 0.25 * math.sqrt(35 / (2 * pi)), 0.5 * math.sqrt(105 / pi), 0.25 * math.sqrt(21 / (2 * pi))
        basis += [-a * y * (3 * x * x - y * y), b * x * y * z, -c * y * (5 * z * z - 1),
                  0.25 * math.sqrt(7 / pi) * z * (5 * z * z - 3), -c * x * (5 * z * z - 1),
                  0.5 * b * z * (x * x - y * y), -a * x * (x * x - 3 * y * y)]
    if degree > 3:
        z2 = z * z
        a, b = 0.75 * math.sqrt(35 / pi), 0.75 * math.sqrt(35 / (2 * pi))
        c, e = 0.75 * math.sqrt(5 / pi), 0.75 * math.sqrt(5 / (2 * pi))
        basis += [a * x * y * (x * x - y * y), -b * y * z * (3 * x * x - y * y), c * x * y * (7 * z2 - 1),
                  -e * y * z * (7 * z2 - 3), 3 / (16 * math.sqrt(pi)) * (35 * z2 * z2 - 30 * z2 + 3),
                  -e * x * z * (7 * z2 - 3), 0.5 * c * (x * x - y * y) * (7 * z2 - 1),
                  -b * x * z * (x * x - 3 * y * y),
                  0.25 * a * (x * x * (x * x - 3 * y * y) - y * y * (3 * x * x - y * y))]
    return (torch.stack(basis, -1)[..., None] * coeffs).sum(-2)


def _tile_lists64(case, proj):
    """Entries (image * tiles + tile, image * n + Gaussian) in tile, then depth
    order, and each tile's first entry."""
    tw, th = -(-case["width"] // TILE), -(-case["height"] // TILE)
    m2, radii = proj["means2d"].reshape(-1, 2), proj["radii"].reshape(-1, 2)
    depth = proj["depths"].reshape(-1)
    grid = torch.tensor([tw, th], device=m2.device)
    low = torch.minimum(torch.floor((m2 - radii) / TILE).long().clamp(min=0), grid)
    high = torch.minimum(torch.ceil((m2 + radii) / TILE).long().clamp(min=0), grid)
    span = torch.where((radii > 0).all(-1, keepdim=True), (high - low).clamp(min=0), torch.zeros_like(low))
    count = span[:, 0] * span[:, 1]
    order = torch.argsort(depth, stable=True)
    order = order[count[order] > 0]
    rows = torch.repeat_interleave(order, count[order])
    start = torch.cumsum(count[order], 0) - count[order]
    k = torch.arange(rows.numel(), device=rows.device) - torch.repeat_interleave(start, count[order])
    w = span[rows, 0]
    tile = (low[rows, 1] + k // w) * tw + low[rows, 0] + k % w + (rows // case["n"]) * (tw * th)
    tile, perm = torch.sort(tile, stable=True)
    first = torch.searchsorted(tile, torch.arange(case["cameras"] * tw * th + 1, device=tile.device))
    return rows[perm], first


def _composite64(case, proj, colors, opacities, background, image_grad=None):
    """The images [C, H, W, 3] and alphas; with image_grad (a function of the
    images) also the gradients of means2d, conics, colors and opacities."""
    W, H, C = case["width"], case["height"], case["cameras"]
    tw, th = -(-W // TILE), -(-H // TILE)
    rows, first = _tile_lists64(case, proj)
    length = first[1:] - first[:-1]
    image = torch.full((C * th * tw, TILE * TILE, 3), background, dtype=torch.float64, device="cuda")
    alpha = torch.zeros((C * th * tw, TILE * TILE, 1), dtype=torch.float64, device="cuda")
    flat = [t.detach().reshape(C * case["n"], -1) for t in (proj["means2d"], proj["conics"], colors, opacities)]
    sums = [torch.zeros_like(t) for t in flat]
    order = torch.argsort(length, descending=True)
    sizes = length[order].tolist()
    chunks, at = [], 0
    while at < len(sizes) and sizes[at] > 0:
        take = max(1, (1 << 24) // (sizes[at] * TILE * TILE))
        chunks.append((order[at : at + take], sizes[at]))
        at += take
    lane = torch.arange(TILE * TILE, device="cuda")

    def blend(tiles, longest, leaves):
        k = torch.arange(longest, device="cuda")
        inside = k[None] < length[tiles][:, None]
        ids = rows[(first[:-1][tiles][:, None] + k[None]).clamp(max=rows.numel() - 1)]
        m2, conic, col, opac = [t[ids] for t in leaves]
        px = (tiles % tw * TILE)[:, None] + lane[None] % TILE + 0.5
        py = (tiles // tw % th * TILE)[:, None] + lane[None] // TILE + 0.5
        dx = m2[:, None, :, 0] - px[..., None]
        dy = m2[:, None, :, 1] - py[..., None]
        sigma = 0.5 * (conic[:, None, :, 0] * dx * dx + conic[:, None, :, 2] * dy * dy) + conic[:, None, :, 1] * dx * dy
        a = torch.clamp(opac[:, None, :, 0] * torch.exp(-sigma), max=0.99)
        a = torch.where((sigma >= 0) & (a >= 1 / 255) & inside[:, None], a, torch.zeros_like(a))
        after = torch.cumsum(torch.log1p(-a), -1)
        a = torch.where(after > math.log(1e-4), a, torch.zeros_like(a))
        log_t = torch.log1p(-a)
        total = torch.cumsum(log_t, -1)
        weight = a * torch.exp(total - log_t)
        T = torch.exp(total[..., -1:])
        return weight @ col + T * background, 1 - T

    with torch.no_grad():
        for tiles, longest in chunks:
            image[tiles], alpha[tiles] = blend(tiles, longest, flat)

    def untile(t):
        t = t.reshape(C, th, tw, TILE, TILE, -1).permute(0, 1, 3, 2, 4, 5)
        return t.reshape(C, th * TILE, tw * TILE, -1)[:, :H, :W].contiguous()

    out, out_alpha = untile(image), untile(alpha)
    if image_grad is None:
        return out, out_alpha
    g = F.pad(image_grad(out), (0, 0, 0, tw * TILE - W, 0, th * TILE - H))
    g = g.reshape(C, th, TILE, tw, TILE, 3).permute(0, 1, 3, 2, 4, 5).reshape(C * th * tw, TILE * TILE, 3)
    for tiles, longest in chunks:
        leaves = [t.requires_grad_(True) for t in flat]
        with torch.enable_grad():
            loss = (blend(tiles, longest, leaves)[0] * g[tiles]).sum()
            for s, d in zip(sums, torch.autograd.grad(loss, leaves)):
                s += d
    return out, out_alpha, [s.reshape(t.shape) for s, t in zip(sums, (proj["means2d"], proj["conics"], colors,
                                                                      opacities))]


def _loss64(case, image, target):
    l1 = (image - target).abs().mean()
    if case.get("loss", "l1") == "l1":
        return l1
    # the trainer's box window is built in the images' float32
    weight = float(np.float32(1.0) / np.float32(SSIM_WINDOW * SSIM_WINDOW))
    pad = SSIM_WINDOW // 2

    def mean(a):
        a = F.pad(a, (0, 0, pad, pad, pad, pad))
        a = a.unfold(1, SSIM_WINDOW, 1).sum(-1)
        return a.unfold(2, SSIM_WINDOW, 1).sum(-1) * weight

    c1, c2 = 0.01**2, 0.03**2
    mx, my = mean(image), mean(target)
    sxx, syy, sxy = mean(image * image) - mx * mx, mean(target * target) - my * my, mean(image * target) - mx * my
    ssim = ((2 * mx * my + c1) * (2 * sxy + c2)) / ((mx * mx + my * my + c1) * (sxx + syy + c2)).clamp(min=1e-12)
    return (1 - SSIM_LAMBDA) * l1 + SSIM_LAMBDA * (1 - ssim.mean()) / 2


def exact(case, seed):
    kind = case["kind"]
    if kind == "lists" or (kind in ("view_sh", "train_sh") and (case["scene"] == "dense" or case["cameras"] > 1 and
                                                                case["n"] * case["cameras"] > 2_500_000)):
        return None
    state = prepare(case, seed)
    if kind == "harmonics":
        dirs, coeffs = [state[k].detach().double().requires_grad_(True) for k in ("dirs", "coeffs")]
        colors = _harmonics64(case["degree"], dirs, coeffs)
        grads = torch.autograd.grad(colors, [dirs, coeffs], state["v_colors"].double(), allow_unused=True)
        return [colors.detach(), grads[0] if grads[0] is not None else torch.zeros_like(dirs), grads[1]]
    train = kind not in ("view_rgb", "view_sh")
    p = {k: v.detach()[0].double().requires_grad_(train) for k, v in state["params"].items()}
    views, Ks = state["viewmats"][0].double(), state["Ks"][0].double()
    if kind == "project":
        out = _project64(case, p["means"], p["quats"], p["scales"], views, Ks, 100.0, model=case["model"])
        names = ["means2d", "depths", "conics"] + (["compensations"] if case["compensations"] else [])
        leaves = [p[k] for k in ("means", "quats", "scales")]
        grads = torch.autograd.grad([out[k] for k in names], leaves,
                                    [c[0].double() for c in state["cotangents"][: len(names)]])
        return [None] + [out[k].detach()[None] for k in names] + [g[None] for g in grads]
    scene = SCENES[case["scene"]]
    C = case["cameras"]
    quats = p["quats"] / p["quats"].norm(dim=-1, keepdim=True)
    opacity = torch.sigmoid(p["opacity_logits"])
    proj = _project64(case, p["means"], quats, torch.exp(p["log_scales"]), views, Ks, scene["far"],
                      opacity if kind == "view_rgb" else None)
    if "degree" in case:
        active = (case["degree"] + 1) ** 2
        coeffs = torch.cat([p["features_dc"][:, None], p["features_rest"][:, : active - 1]], 1)
        centres = [-(views[c, :3, :3].T @ views[c, :3, 3]) for c in range(C)]
        colors = torch.stack([torch.clamp(_harmonics64(case["degree"], p["means"] - o, coeffs) + 0.5, 0, 1)
                              for o in centres])
    else:
        colors = p["colors"].expand(C, -1, -1)
    opac = opacity.expand(C, -1)
    if not train:
        return list(_composite64(case, proj, colors, opac, scene["bg"]))
    target = state["target"].double()
    value = {}

    def image_grad(image):
        image = image.requires_grad_(True)
        with torch.enable_grad():
            value["loss"] = _loss64(case, image, target)
        return torch.autograd.grad(value["loss"], image)[0]

    image, alpha, grads = _composite64(case, proj, colors, opac, scene["bg"], image_grad)
    leaves = list(p.values())
    out = torch.autograd.grad([proj["means2d"], proj["conics"], colors, opac], leaves, grads, allow_unused=True)
    out = [(g if g is not None else torch.zeros_like(leaf))[None] for g, leaf in zip(out, leaves)]
    result = [value["loss"].detach(), image.detach(), alpha]
    return result + out if kind == "fit_rgb" else result + out + [grads[0][None]]
