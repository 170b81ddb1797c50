"""The renderer's performance cases: frames, prefilters and training steps over the sizes this framework is used at.

Six kinds of call, each through the public entry point that a program uses:

  frame          GaussianRasterizer under torch.no_grad(): one rendered view, activated Gaussians in hand
  filter         GaussianRasterizer.visible_filter: the visibility prefilter of a scene
  train          GaussianModel in training mode: forward from the raw parameters, backward to their gradients
  anchors        ScaffoldGS in evaluation mode: prefilter, anchor decode and rasterizer of one view
  octree         OctreeGS in evaluation mode: the same behind a level-of-detail mask
  anchor_train   ScaffoldGS in training mode: forward and backward to the anchors' and the decoder's gradients

Scenes are synthetic, drawn on the GPU from the seed with the distributions of landmarksystem_amd/scenes.py:

  ball   an object: Gaussians ~ N(0, 5^2), camera at distance 20 (config2)
  slab   a city block 200 m x 200 m seen whole by an aerial camera (config3, config5)
  part   a district 600 m x 600 m of which the camera sees a fifth to three fifths (config4)

The size of a splat follows the number of Gaussians, so that a scene of fewer of them covers the same area: early in
training a scene holds few, large Gaussians, late in training many small ones.
"""
import math
import random

import torch

from landmarksystem_amd import GaussianRasterizationSettings, GaussianRasterizer, scenes
from landmarksystem_amd.cameras import Camera
from landmarksystem_amd.models import GaussianModel, OctreeGS, ScaffoldGS

# scene -> (Gaussians at which its mean log scale holds, that mean, its spread, opacity logit mean,
#           share of the Gaussians that a view keeps, (pixel, Gaussian) pairs per pixel that a view blends)
_SCENES = {
    "ball": (1_000_000, -3.0, 0.7, 0.0, 0.95, 120),
    "slab": (6_000_000, -2.5, 0.8, 0.5, 0.88, 50),
    "part": (20_000_000, -2.5, 0.8, 0.5, 0.40, 30),
}
_N_OFFSETS, _FEAT_DIM = 10, 32


def listed():
    return [
        # the smallest call: a preview of a sparse reconstruction, where launches and host work are all there is (config1)
        dict(name="frame_10k_256", kind="frame", scene="ball", gaussians=10_000, width=256, height=256, sh_degree=0,
             precomputed=False),
        # colours and covariances evaluated by the caller (override_color, compute_cov3D_python), image size off the
        # tile grid, Gaussian count off every block size
        dict(name="frame_130k_ragged", kind="frame", scene="slab", gaussians=130_003, width=979, height=546, sh_degree=1,
             precomputed=True),
        # an object filling the view: large splats, many (tile, Gaussian) pairs per Gaussian (config2)
        dict(name="frame_1m_1080p", kind="frame", scene="ball", gaussians=1_000_000, width=1920, height=1080,
             sh_degree=3, precomputed=False),
        # the benchmark's default view (config3)
        dict(name="frame_6m_1080p", kind="frame", scene="slab", gaussians=6_000_000, width=1920, height=1080,
             sh_degree=3, precomputed=False),
        # a view of a 4K trajectory over a large scene, most of it culled (config4)
        dict(name="frame_20m_4k", kind="frame", scene="part", gaussians=20_000_000, width=3840, height=2160,
             sh_degree=3, precomputed=False),
        # the prefilter on its own: which Gaussians does this view need (block loading, the models' prefilter_voxel)
        dict(name="filter_6m_1080p", kind="filter", scene="part", gaussians=6_000_000, width=1920, height=1080),
        # a training step soon after initialisation from a point cloud, spherical harmonics still growing
        dict(name="train_100k_ragged", kind="train", scene="ball", gaussians=100_003, width=801, height=533,
             sh_degree=2),
        # a training step at full size
        dict(name="train_6m_1080p", kind="train", scene="slab", gaussians=6_000_000, width=1920, height=1080,
             sh_degree=3),
        # small anchor scene, odd sizes
        dict(name="anchors_60k_ragged", kind="anchors", anchors=60_001, width=1237, height=823, bank=False),
        # the benchmark's anchor scene, with the fp32 weights and features of a trained checkpoint (config5)
        dict(name="anchors_500k_1080p", kind="anchors", anchors=500_000, width=1920, height=1080, bank=False),
        # level of detail over a larger anchor scene, feature bank on
        dict(name="octree_1m_1080p", kind="octree", anchors=1_000_000, width=1920, height=1080, bank=True),
        # a training step through the anchor decode
        dict(name="anchor_train_200k_1080p", kind="anchor_train", anchors=200_000, width=1920, height=1080, bank=False),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(("frame", "frame", "frame", "filter", "train", "train", "anchors", "octree", "anchor_train"))
    small = kind in ("train", "anchor_train")
    width = _log_uniform(rng, 200, 1920 if small else 3200)
    case = dict(kind=kind, width=width, height=max(16, int(width * rng.uniform(0.5, 1.0))))
    if kind in ("frame", "filter", "train"):
        case["scene"] = rng.choice(("ball", "slab", "part"))
        case["gaussians"] = _log_uniform(rng, 5_000, {"frame": 10_000_000, "filter": 12_000_000, "train": 4_000_000}[kind])
        if kind != "filter":
            case["sh_degree"] = rng.choice((0, 1, 2, 3, 3))
        if kind == "frame":
            case["precomputed"] = rng.random() < 0.25
    else:
        case["anchors"] = _log_uniform(rng, 5_000, 300_000 if small else 1_200_000)
        case["bank"] = rng.random() < 0.3
    return case


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _slab_points(n, half_extent, g):
    xy = (torch.rand(n, 2, generator=g, device=g.device) * 2 - 1) * half_extent
    z = (-5.0 * torch.log(torch.rand(n, 1, generator=g, device=g.device).clamp_min(1e-12))).clamp(0.0, 40.0)
    return torch.cat([xy, z], dim=1)


def _unit_quaternions(n, g):
    return torch.nn.functional.normalize(torch.randn(n, 4, generator=g, device=g.device))


def _camera(scene, width, height, points, seed):
    """A view of the scene that differs from seed to seed, as the views of a trajectory or a training set do."""
    rng = random.Random(seed)
    if scene == "part":
        cpu = torch.Generator().manual_seed(seed)
        return scenes.aerial_poses(1, width, height, cpu, points=points[:20_000].cpu())[0].to(points.device)
    yaw = rng.uniform(0.0, 2.0 * math.pi)
    if scene == "ball":
        up = rng.uniform(-0.5, 0.5)
        eye = [20.0 * math.cos(up) * math.cos(yaw), 20.0 * math.cos(up) * math.sin(yaw), 20.0 * math.sin(up)]
    else:
        eye = [150.0 * math.cos(yaw), 150.0 * math.sin(yaw), 150.0]
    return Camera.look_at(eye, [0.0, 0.0, 0.0], [0.0, 0.0, 1.0], width, height, math.radians(60.0)).to(points.device)


def _settings(camera, sh_degree):
    return GaussianRasterizationSettings(
        image_height=camera.height, image_width=camera.width, tanfovx=math.tan(camera.FovX * 0.5),
        tanfovy=math.tan(camera.FovY * 0.5), bg=torch.zeros(3, device=camera.device), scale_modifier=1.0,
        viewmatrix=camera.world_view_transform, projmatrix=camera.full_proj_transform, sh_degree=sh_degree,
        campos=camera.camera_center, prefiltered=False, debug=False)


def _covariance(scales, q):
    r, x, y, z = q.unbind(1)
    R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - r * z), 2 * (x * z + r * y),
                     2 * (x * y + r * z), 1 - 2 * (x * x + z * z), 2 * (y * z - r * x),
                     2 * (x * z - r * y), 2 * (y * z + r * x), 1 - 2 * (x * x + y * y)], dim=1).view(-1, 3, 3)
    L = R * scales[:, None, :]
    S = torch.stack([(L[:, a] * L[:, b]).sum(dim=1) for a, b in ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))], dim=1)
    return S.contiguous()


def _anchor_model(case, g):
    A = case["anchors"]
    dev = g.device
    rand = lambda *shape: torch.randn(*shape, generator=g, device=dev)  # noqa: E731
    anchor = _slab_points(A, 100.0, g)
    log_scale = rand(A, 6) * 0.8 - 2.5 + 0.5 * math.log(500_000 / A)
    rotation = torch.zeros(A, 4, device=dev)
    rotation[:, 0] = 1.0
    octree = case["kind"] == "octree"
    kw = dict(n_offsets=_N_OFFSETS, use_feat_bank=case["bank"], act_cache=case["kind"] != "anchor_train")
    args = (anchor, rand(A, _FEAT_DIM) * 0.5, rand(A, _N_OFFSETS, 3) * 0.1, log_scale, rotation)
    if octree:
        level = torch.randint(0, 5, (A,), generator=g, device=dev).float()
        model = OctreeGS(*args, level, voxel_size=0.5, standard_dist=250.0, add_opacity_dist=False, add_cov_dist=False,
                         add_color_dist=False, **kw)
    else:
        model = ScaffoldGS(*args, **kw)
    model = model.to(dev)
    with torch.no_grad():
        for p in model.anchor_decoder.parameters():
            p.copy_(rand(*p.shape) * (p.shape[1] ** -0.5 if p.dim() == 2 else 0.05))
    return model


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind, width, height = case["kind"], case["width"], case["height"]
    state = {"kind": kind}
    if kind in ("anchors", "octree", "anchor_train"):
        model = _anchor_model(case, g)
        state.update(model=model, camera=_camera("slab", width, height, model.get_anchor, seed))
        if kind == "anchor_train":
            model.train()
            leaves = [model._anchor_feat, model._offset, model._scaling] + list(model.anchor_decoder.parameters())
            for p in leaves:
                p.requires_grad_(True)
            state.update(leaves=leaves, cotangent=torch.randn(3, height, width, generator=g, device="cuda") / (height * width),
                         reg_weight=torch.tensor(0.01, device="cuda"))
        else:
            model.eval()
        return state
    P = case["gaussians"]
    base, log_mean, log_spread, logit_mean, _, _ = _SCENES[case["scene"]]
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")  # noqa: E731
    if case["scene"] == "ball":
        means = rand(P, 3) * 5.0
    else:
        means = _slab_points(P, 100.0 if case["scene"] == "slab" else 300.0, g)
    log_scales = rand(P, 3) * log_spread + (log_mean + 0.5 * math.log(base / P))
    log_scales = torch.maximum(log_scales, log_scales.max(dim=1, keepdim=True).values - math.log(50.0))
    rotations = _unit_quaternions(P, g)
    state["camera"] = camera = _camera(case["scene"], width, height, means, seed)
    if kind == "filter":
        state.update(rasterizer=GaussianRasterizer(_settings(camera, 1)),
                     inputs=dict(means3D=means, scales=torch.exp(log_scales), rotations=rotations))
        return state
    logits = rand(P, 1) * 1.5 + logit_mean
    coeffs = (case["sh_degree"] + 1) ** 2
    dc, rest = rand(P, 1, 3) * 0.3, rand(P, coeffs - 1, 3) * 0.05
    if kind == "train":
        model = GaussianModel(means, dc, rest, log_scales, rotations * (0.5 + torch.rand(P, 1, generator=g, device="cuda")),
                              logits, sh_degree=case["sh_degree"]).cuda().train()
        leaves = [model._xyz, model._features_dc, model._features_rest, model._scaling, model._rotation, model._opacity]
        for p in leaves:
            p.requires_grad_(True)
        state.update(model=model, leaves=leaves, cotangent=rand(3, height, width) / (height * width))
        return state
    inputs = dict(means3D=means, means2D=None, opacities=torch.sigmoid(logits), shs=None, colors_precomp=None,
                  scales=None, rotations=None, cov3D_precomp=None)
    if case["precomputed"]:
        inputs.update(colors_precomp=torch.rand(P, 3, generator=g, device="cuda"),
                      cov3D_precomp=_covariance(torch.exp(log_scales), rotations))
    else:
        inputs.update(shs=torch.cat([dc, rest], dim=1), scales=torch.exp(log_scales), rotations=rotations)
    state.update(rasterizer=GaussianRasterizer(_settings(camera, case["sh_degree"])), inputs=inputs)
    return state


# ---- one pass -------------------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "frame":
        rasterizer = state["rasterizer"]
        with torch.no_grad():
            image, radii, depth = rasterizer(**state["inputs"])
        return {"image": image, "radii": radii, "depth": depth, "alpha": rasterizer.last_alpha}
    if kind == "filter":
        with torch.no_grad():
            return state["rasterizer"].visible_filter(**state["inputs"])
    model = state["model"]
    if kind in ("anchors", "octree"):
        with torch.no_grad():
            image = model(state["camera"])
        return {"image": image, "depth": model.renderer.last_depth, "alpha": model.renderer.last_alpha,
                "anchors": model.voxel_visible_mask}
    leaves = state["leaves"]
    for p in leaves:
        p.grad = None
    if kind == "train":
        image = model(state["camera"])
        image.backward(state["cotangent"])
        # (radii and the screen-space gradient: what densification reads)
        return {"image": image.detach(), "radii": model.radii, "screen": model.viewspace_points.grad,
                "grads": [p.grad for p in leaves]}
    image, scaling = model(state["camera"], retain_grad=True)
    reg = scaling.prod(dim=1).mean()  # the volume regulariser of anchor training
    torch.autograd.backward((image, reg), (state["cotangent"], state["reg_weight"]))
    # what densification accumulates, by anchor and offset: offsets selected, opacities, screen-space gradients
    visible = model.voxel_visible_mask[:, None].expand(-1, _N_OFFSETS).reshape(-1)
    selected = torch.zeros_like(visible).masked_scatter_(visible, model.offset_selection_mask)
    opacity = torch.zeros(visible.shape[0], device=visible.device).masked_scatter_(visible, model.opacity.detach())
    screen = torch.zeros(visible.shape[0], 3, device=visible.device)
    screen.masked_scatter_(selected[:, None], model.viewspace_points.grad)
    return {"image": image.detach(), "reg": reg.detach(), "opacity": opacity, "selected": selected, "screen": screen,
            "grads": [p.grad for p in leaves]}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def work(case):
    """Bytes: each input read once (of a culled Gaussian only what decides that), each output written once.  Flops: the
    anchor decode's products, the blended (pixel, Gaussian) pairs at 25 each (three times that backward)."""
    kind, pixels = case["kind"], case["width"] * case["height"]
    if kind in ("anchors", "octree", "anchor_train"):
        A = case["anchors"]
        seen = A * (0.23 if kind == "octree" else 0.88)
        per_anchor = 4 * (3 + _FEAT_DIM + 3 * _N_OFFSETS + 6)
        flops = seen * 2 * (3 * 36 * 32 + 32 * 110) + 25 * 20 * pixels
        nbytes = A * 44 + seen * per_anchor + 20 * pixels + A
        if kind == "anchor_train":
            return {"bytes": A * 44 + seen * per_anchor + 4 * A * (_FEAT_DIM + 3 * _N_OFFSETS + 6)
                    + seen * _N_OFFSETS * (4 + 1 + 12) + 4 * 6 * pixels, "flops": 3 * flops}
        return {"bytes": nbytes, "flops": flops}
    P = case["gaussians"]
    if kind == "filter":
        return {"bytes": P * (40 + 4), "flops": P * 150}
    _, _, _, _, share, pairs = _SCENES[case["scene"]]
    coeffs = (case["sh_degree"] + 1) ** 2
    rest = 4 * (6 + 3 + 1) if case.get("precomputed") else 4 * (3 + 4 + 1 + 3 * coeffs)
    flops = 25 * pairs * pixels
    if kind == "train":
        parameters = 4 * (3 + 3 + 4 + 1 + 3 * coeffs)
        return {"bytes": P * 12 + P * share * rest + P * (parameters + 12 + 4) + 4 * 6 * pixels, "flops": 4 * flops}
    return {"bytes": P * 12 + P * share * rest + P * 4 + 20 * pixels, "flops": flops}


def tolerance(case):
    """fp32 sums throughout.  `max` is wider than `rel` asks for: a pixel takes or leaves a Gaussian at alpha = 1/255,
    so a difference in the last bits of an exponent can move single pixels by that much of a colour, and with them the
    gradient of a Gaussian that few pixels see; whole values are exact but for opacities within rounding of zero."""
    if case["kind"] == "filter":
        return "exact"
    if case["kind"] == "frame":
        return {"rel": 1e-5, "max": 0.02}
    if case["kind"] in ("anchors", "octree"):
        return {"rel": 1e-4, "max": 0.05}
    return {"rel": 1e-4, "max": 0.2, "differ": 1e-5 if case["kind"] == "anchor_train" else 0.0}
