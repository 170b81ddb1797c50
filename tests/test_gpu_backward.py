"""GPU parity of the backward pass: gs355_render_backward (through the C ABI and through autograd) against the
double-precision CPU oracle on identical seeded inputs.

Bar: floating point (fp32 sums of up to thousands of pixel contributions against the oracle's float64).  Every
gradient element must be within 1e-4 of the tensor's largest magnitude plus 1e-3 of the largest component of the same
Gaussian's gradient of the oracle's value (measured: a few 1e-6 of the largest magnitude on the small scenes)."""
import numpy as np
import pytest
import torch

from landmarksystem_amd import GaussianRasterizer, _lib, models, pipeline, scenes
from oracle import c_oracle as co
from tests.helpers import oracle_frame, oracle_gaussians, settings_for

pytestmark = pytest.mark.gpu

ABS_OF_MAX, REL = 1e-4, 1e-3


def assert_grad_close(got, ref, name):
    got = np.asarray(got, np.float64).reshape(ref.shape)
    scale = np.abs(ref).max()
    # components of one Gaussian's gradient come out of the same sums: a small component next to a large one
    # carries the large one's rounding error, so the relative part is taken of the Gaussian's largest component
    row = np.abs(ref).reshape(ref.shape[0], -1).max(axis=1).reshape((-1,) + (1,) * (ref.ndim - 1)) if ref.ndim > 1 \
        else np.abs(ref)
    bound = ABS_OF_MAX * scale + REL * row
    err = np.abs(got - ref)
    worst = np.unravel_index(np.argmax(err - bound), err.shape)
    assert (err <= bound).all(), "%s: element %s differs by %g (value %g, largest magnitude %g)" % (
        name, worst, err[worst], ref[worst], scale)


def cotangents(scene, seed):
    g = torch.Generator().manual_seed(seed)
    H, W = scene.camera.height, scene.camera.width
    return (torch.randn(3, H, W, generator=g), torch.randn(1, H, W, generator=g), torch.randn(1, H, W, generator=g))


def oracle_backward(scene, gi, gd=None, ga=None, colors=None, cov=None, sh_degree=None):
    cf = oracle_frame(scene, sh_degree=sh_degree)
    cg = oracle_gaussians(scene, colors_precomp=None if colors is None else colors.numpy(),
                          cov3D_precomp=None if cov is None else cov.numpy())
    fwd = co.render(cf, cg)
    # Pixels where the forward pass took a discrete decision (alpha < 1/255, T (1 - alpha) < 1e-4) within rounding
    # of its threshold may legitimately decide otherwise on the GPU (the forward parity tests exclude them too):
    # their cotangents are zeroed, IN PLACE, so that the GPU run that follows sees the same loss.
    keep = torch.from_numpy(fwd["fragile"] == 0)
    for t in (gi, gd, ga):
        if t is not None:
            t.mul_(keep)
    return co.render_backward(cf, cg, fwd, gi.numpy(), None if gd is None else gd.numpy()[0],
                              None if ga is None else ga.numpy()[0]), fwd


def abi_backward(scene, device, gi, gd=None, ga=None, colors=None, cov=None, sh_degree=None, want=pipeline.GRAD_NAMES,
                 classic=False):
    """Forward and backward through pipeline.render / pipeline.render_backward (thin ctypes calls of the C ABI)."""
    s = settings_for(scene, device, sh_degree=sh_degree)
    dev = lambda t: None if t is None else t.to(device)  # noqa: E731
    inp = pipeline.FrameInputs(s, dev(scene.means3D), opacities=dev(scene.opacities),
                               shs=None if colors is not None else dev(scene.shs), colors_precomp=dev(colors),
                               scales=None if cov is not None else dev(scene.scales),
                               rotations=None if cov is not None else dev(scene.rotations), cov3D_precomp=dev(cov))
    ws = pipeline.Workspace(device)
    out = pipeline.render(inp, ws=ws, classic=classic)
    grads = pipeline.render_backward(inp, out, ws.buffer, dev(gi), dev(gd), dev(ga), want=want)
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in grads.items()}, out


@pytest.mark.parametrize("deg", [0, 1, 2, 3])
def test_backward_all_sh_degrees(gpu_device, deg):
    scene = scenes.tiny_scene(P=400, width=100, height=70, sh_degree=deg, seed=3 + deg)
    gi, gd, ga = cotangents(scene, deg)
    ref, _ = oracle_backward(scene, gi, gd, ga)
    got, _ = abi_backward(scene, gpu_device, gi, gd, ga)
    assert set(got) == {"means3D", "means2D", "shs", "opacities", "scales", "rotations"}
    for name, value in got.items():
        assert_grad_close(value, ref[name], "deg %d %s" % (deg, name))


def test_backward_with_precomputed_colours_and_covariances(gpu_device):
    scene = scenes.tiny_scene(P=400, width=100, height=70, sh_degree=0, seed=9)
    g = torch.Generator().manual_seed(1)
    colors = torch.rand(scene.P, 3, generator=g)
    cov = torch.from_numpy(np.stack([co.cov3d(scene.scales[i].numpy(), 1.0, scene.rotations[i].numpy())
                                     for i in range(scene.P)]))
    gi, gd, ga = cotangents(scene, 2)
    ref, _ = oracle_backward(scene, gi, gd, ga, colors=colors, cov=cov, sh_degree=1)
    got, _ = abi_backward(scene, gpu_device, gi, gd, ga, colors=colors, cov=cov, sh_degree=1)
    assert set(got) == {"means3D", "means2D", "colors_precomp", "opacities", "cov3D_precomp"}
    for name, value in got.items():
        assert_grad_close(value, ref[name], name)


def test_backward_image_gradient_only_and_selected_outputs(gpu_device):
    """The training loop's case: a loss on the image alone; only some gradients requested."""
    scene = scenes.config1()
    gi, _, _ = cotangents(scene, 5)
    ref, _ = oracle_backward(scene, gi)
    got, _ = abi_backward(scene, gpu_device, gi, want=("means3D", "opacities", "means2D"))
    assert set(got) == {"means3D", "opacities", "means2D"}
    for name, value in got.items():
        assert_grad_close(value, ref[name], name)


@pytest.mark.parametrize("make,label", [
    (lambda: scenes.config3(P=100_000, width=480, height=270), "C3/100k at 480x270"),
    (lambda: scenes.config2(P=60_000, width=333, height=177), "C2/60k ragged image"),
])
def test_backward_scaled_down_configs(gpu_device, make, label):
    scene = make()
    gi, gd, ga = cotangents(scene, 8)
    ref, fwd = oracle_backward(scene, gi, gd, ga)
    got, out = abi_backward(scene, gpu_device, gi, gd, ga)
    assert out.num_keys == fwd["num_keys"]
    culled = fwd["radii"] == 0
    assert culled.any()
    for name, value in got.items():
        assert_grad_close(value, ref[name], label + " " + name)
        assert (value[culled] == 0).all(), name  # written, not left uninitialised


def test_backward_of_a_crowded_tile_with_finished_pixels(gpu_device):
    """Thousands of Gaussians over one small image: several staged batches per tile, pixels that reach the
    1e-4 transmittance stop, and every Gaussian beyond the stop gets a zero gradient."""
    scene = scenes.tiny_scene(P=3000, width=48, height=48, sh_degree=1, seed=31, spread=0.3, log_scale_mean=-1.2)
    gi, gd, ga = cotangents(scene, 3)
    ref, fwd = oracle_backward(scene, gi, gd, ga)
    got, _ = abi_backward(scene, gpu_device, gi, gd, ga)
    assert fwd["alpha"].max() > 0.9998
    untouched = np.abs(ref["acc"]).sum(1) == 0
    assert (untouched & (fwd["radii"] > 0)).sum() > 100
    for name, value in got.items():
        assert_grad_close(value, ref[name], name)
    assert (got["opacities"][untouched] == 0).all()


def test_autograd_through_the_rasterizer(gpu_device):
    """GaussianRasterizer called as the reference's training loop calls it: gradients arrive on the leaves,
    `means2D` carries the screen-space gradient, non-contiguous inputs get gradients of their own shape."""
    scene = scenes.tiny_scene(P=500, width=96, height=64, sh_degree=2, seed=17)
    gi, gd, ga = cotangents(scene, 1)
    ref, _ = oracle_backward(scene, gi, gd, ga)
    leaf = lambda t: t.to(gpu_device).clone().requires_grad_(True)  # noqa: E731
    means, opac, shs, rots = leaf(scene.means3D), leaf(scene.opacities), leaf(scene.shs), leaf(scene.rotations)
    scales6 = leaf(torch.cat([scene.scales, torch.ones(scene.P, 3)], 1))  # the models pass a strided [:, :3] slice
    means2D = torch.zeros_like(means, requires_grad=True) + 0
    means2D.retain_grad()
    r = GaussianRasterizer(settings_for(scene, gpu_device))
    image, radii, depth = r(means3D=means, means2D=means2D, shs=shs, colors_precomp=None, opacities=opac,
                            scales=scales6[:, :3], rotations=rots, cov3D_precomp=None)
    assert image.requires_grad and depth.requires_grad and r.last_alpha.requires_grad and not radii.requires_grad
    loss = (image * gi.to(gpu_device)).sum() + (depth * gd.to(gpu_device)).sum() + (r.last_alpha * ga.to(gpu_device)).sum()
    loss.backward()
    assert opac.grad.shape == opac.shape and scales6.grad.shape == scales6.shape
    assert (scales6.grad[:, 3:] == 0).all()
    for name, value in (("means3D", means.grad), ("means2D", means2D.grad), ("opacities", opac.grad), ("shs", shs.grad),
                        ("scales", scales6.grad[:, :3]), ("rotations", rots.grad)):
        assert_grad_close(value.cpu().numpy(), ref[name], name)
    # a second frame on the same stream before the first one's backward pass must not disturb it
    image1, _, _ = r(means3D=means, means2D=None, shs=shs, colors_precomp=None, opacities=opac,
                     scales=scales6[:, :3], rotations=rots, cov3D_precomp=None)
    other = scenes.tiny_scene(P=200, width=96, height=64, sh_degree=2, seed=18)
    with torch.no_grad():
        r(means3D=other.means3D.to(gpu_device), shs=other.shs.to(gpu_device), opacities=other.opacities.to(gpu_device),
          scales=other.scales.to(gpu_device), rotations=other.rotations.to(gpu_device))
    means.grad = None
    (image1 * gi.to(gpu_device)).sum().backward()
    ref_image_only, _ = oracle_backward(scene, gi)
    assert_grad_close(means.grad.cpu().numpy(), ref_image_only["means3D"], "means3D after an interleaved frame")


def test_no_grad_call_is_the_plain_forward(gpu_device):
    scene = scenes.tiny_scene(P=100, width=64, height=48, sh_degree=1, seed=2)
    means = scene.means3D.to(gpu_device).requires_grad_(True)
    r = GaussianRasterizer(settings_for(scene, gpu_device))
    with torch.no_grad():
        image, _, _ = r(means3D=means, shs=scene.shs.to(gpu_device), opacities=scene.opacities.to(gpu_device),
                        scales=scene.scales.to(gpu_device), rotations=scene.rotations.to(gpu_device))
    assert not image.requires_grad


def test_training_step_of_the_vanilla_model(gpu_device):
    """The reference's training forward (origin_gs/gs_model.py:112-228): all Gaussians rendered, the screen-space
    points kept for densification; one backward pass fills the parameters' gradients."""
    scene = scenes.tiny_scene(P=600, width=96, height=64, sh_degree=3, seed=23)
    model = models.GaussianModel.from_activated(scene.means3D, scene.scales, scene.rotations, scene.opacities,
                                                scene.shs, fuse_prefilter=False).to(gpu_device)
    for p in model.parameters():
        p.requires_grad_(True)
    model.train()
    image = model(scene.camera)
    assert image.requires_grad
    target = torch.rand_like(image)
    loss = (image - target).abs().mean()
    loss.backward()
    assert model.viewspace_points.grad is not None
    vis = model.visibility_filter
    assert (model.viewspace_points.grad[vis, :2].norm(dim=-1) > 0).any()
    assert (model.viewspace_points.grad[~vis] == 0).all()
    for name, p in model.named_parameters():
        assert p.grad is not None and torch.isfinite(p.grad).all(), name
    assert model._xyz.grad.abs().max() > 0 and model._features_rest.grad.abs().max() > 0
    assert model.radii.shape[0] == scene.P  # training: no gather, radii of every Gaussian (what densification indexes)
    # the single-pass variant (no separate visibility prefilter) leaves the same by-products and gradients
    fused = models.GaussianModel.from_activated(scene.means3D, scene.scales, scene.rotations, scene.opacities,
                                                scene.shs, fuse_prefilter=True).to(gpu_device).train()
    for p in fused.parameters():
        p.requires_grad_(True)
    image2 = fused(scene.camera)
    (image2 - target).abs().mean().backward()
    assert torch.equal(image2, image) and torch.equal(fused.visibility_filter, vis)
    assert torch.equal(fused.radii, model.radii)
    torch.testing.assert_close(fused._xyz.grad, model._xyz.grad, rtol=1e-4, atol=1e-6 * float(model._xyz.grad.abs().max()))
    torch.testing.assert_close(fused.viewspace_points.grad, model.viewspace_points.grad, rtol=1e-4,
                               atol=1e-6 * float(model.viewspace_points.grad.abs().max()))


def test_full_size_headline_frame_backward_equals_the_oracle(gpu_device):
    """The 6M-Gaussian 1080p frame: every gradient of an image loss against the oracle's backward pass (all host
    cores, about a quarter of a minute), and two runs of the kernels against each other.  Sums run in a fixed order
    except inside a tile's batch, where the rows' totals reach a key's accumulators in the order the hardware serves
    them: last bits of the per-key records move, and a thin splat's scale gradient amplifies them (measured over
    eight pairs of runs: up to 1e-5 of the tensor's largest magnitude for scales, 1e-6 or less elsewhere)."""
    scene = scenes.config3()
    gi, _, _ = cotangents(scene, 11)
    ref, fwd = oracle_backward(scene, gi)
    got, out = abi_backward(scene, gpu_device, gi)
    assert out.num_keys == fwd["num_keys"] > 10_000_000
    for name, value in got.items():
        assert_grad_close(value, ref[name], "6M " + name)
    again, _ = abi_backward(scene, gpu_device, gi)
    for name, value in got.items():
        scale = np.abs(value).max()
        assert np.abs(value - again[name]).max() <= 1e-4 * scale, name  # (the bar of the comparison with the oracle)


@pytest.mark.parametrize("classic", [True, False])
def test_backward_after_either_pipeline_on_a_large_image(gpu_device, classic):
    """More than 36000 tiles, forward through scan / duplicate / radix sort / ranges or through the bucketed stages
    (which count per coarse bin at this size): the backward pass reads the same workspace arrays either way."""
    scene = scenes.config2(P=20_000, width=4000, height=2400)  # 250 x 150 = 37500 tiles
    # Splats up to 90 px in radius: thousands of pixels per sum.  Cotangents of one sign, as a smooth loss gives
    # them; with random signs the fp32 sums cancel to 1/100 of their terms and lose the digits the bar asks for.
    gi, gd, _ = (t.abs() for t in cotangents(scene, 4))
    ref, fwd = oracle_backward(scene, gi, gd)
    got, out = abi_backward(scene, gpu_device, gi, gd, classic=classic)
    assert out.num_keys == fwd["num_keys"]
    for name, value in got.items():
        assert_grad_close(value, ref[name], name)


def test_backward_edge_cases(gpu_device):
    """No Gaussians; nothing visible; a one-tile image smaller than a tile."""
    scene = scenes.tiny_scene(P=50, width=9, height=5, sh_degree=1, seed=6)
    gi, gd, ga = cotangents(scene, 0)
    ref, _ = oracle_backward(scene, gi, gd, ga)
    got, _ = abi_backward(scene, gpu_device, gi, gd, ga)
    for name, value in got.items():
        assert_grad_close(value, ref[name], "9x5 " + name)
    # nothing visible: every Gaussian behind the camera
    behind = scenes.tiny_scene(P=50, width=32, height=32, sh_degree=1, seed=6)
    behind.means3D[:, 2] -= 100.0
    gi, gd, ga = cotangents(behind, 0)
    got, out = abi_backward(behind, gpu_device, gi, gd, ga)
    assert out.num_keys == 0
    for name, value in got.items():
        assert (value == 0).all(), name
    # no Gaussians at all
    s = settings_for(behind, gpu_device)
    e = lambda *shape: torch.empty(*shape, device=gpu_device)  # noqa: E731
    inp = pipeline.FrameInputs(s, e(0, 3), opacities=e(0, 1), shs=e(0, 4, 3), scales=e(0, 3), rotations=e(0, 4))
    ws = pipeline.Workspace(gpu_device)
    out = pipeline.render(inp, ws=ws)
    grads = pipeline.render_backward(inp, out, ws.buffer, gi.to(gpu_device))
    torch.cuda.synchronize()
    assert all(v.numel() == 0 for v in grads.values())


def test_gradient_descent_through_the_model_fits_a_target(gpu_device):
    """End to end, as the reference's trainer uses the rasterizer (origin_gs/gs_trainer.py:117-137): a perturbed copy
    of a scene is optimised with Adam against the original's rendering; the L1 loss must fall by more than half."""
    scene = scenes.tiny_scene(P=400, width=96, height=64, sh_degree=1, seed=41, log_scale_mean=-1.8)
    make = lambda s: models.GaussianModel.from_activated(s.means3D, s.scales, s.rotations, s.opacities, s.shs,  # noqa: E731
                                                         sh_degree=1).to(gpu_device)
    with torch.no_grad():
        target = make(scene).eval()(scene.camera)
    g = torch.Generator().manual_seed(0)
    scene.means3D += 0.03 * torch.randn(scene.P, 3, generator=g)
    scene.shs += 0.1 * torch.randn(scene.shs.shape, generator=g)
    scene.scales *= torch.exp(0.2 * torch.randn(scene.P, 3, generator=g))
    model = make(scene).train()
    for p in model.parameters():
        p.requires_grad_(True)
    opt = torch.optim.Adam(model.parameters(), lr=5e-3)
    losses = []
    for _ in range(60):
        loss = (model(scene.camera) - target).abs().mean()
        opt.zero_grad(set_to_none=True)
        loss.backward()
        opt.step()
        losses.append(float(loss.detach()))
    assert losses[-1] < 0.5 * losses[0], (losses[0], losses[-1])
    assert all(np.isfinite(losses))


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("where", ["colour", "cotangent"])
def test_values_that_are_not_finite_reach_the_gaussians_of_their_pixels_only(gpu_device, where, value):
    """A colour or a pixel's cotangent that is not finite: the gradients that the pixels concerned feed are not finite, all
    others are the same bits as without it (four list entries share the reduction over a block's pixels)."""
    scene = scenes.tiny_scene(P=400, width=133, height=75, sh_degree=0, seed=3)
    colours = torch.rand(400, 3, generator=torch.Generator().manual_seed(0))
    gi, gd, ga = cotangents(scene, 4)

    def grads(colours, gi, gd=gd, ga=ga):
        got, out = abi_backward(scene, gpu_device, gi, gd, ga, colors=colours)
        return got, out.image.cpu()

    want, image = grads(colours, gi)
    bad_colours, bad_gi = colours.clone(), gi.clone()
    if where == "colour":
        bad_colours[17] = 2.0
        touched = (grads(bad_colours, gi)[1] != image).any(dim=0)
        bad_colours[17] = value
    else:
        touched = torch.zeros(75, 133, dtype=torch.bool)
        touched[41, 70] = True
        bad_gi[:, 41, 70] = value
    assert 0 < int(touched.sum()) < touched.numel() // 2
    # the Gaussians that blend in those pixels: the weights are positive, so a cotangent of ones leaves no gradient zero
    zero = torch.zeros_like(gd)
    there, _ = grads(colours, touched.float().expand(3, -1, -1).contiguous(), zero, zero)
    concerned = there["colors_precomp"].any(axis=1)
    assert 0 < concerned.sum() < 200
    got, _ = grads(bad_colours, bad_gi)
    for name in ("opacities", "means3D", "means2D", "scales") + (("colors_precomp",) if where == "cotangent" else ()):
        finite = np.isfinite(got[name].reshape(400, -1))
        assert not finite[concerned].all(axis=1).any(), name
        assert finite[~concerned].all(), name
    for name, value in got.items():
        assert np.array_equal(value.reshape(400, -1)[~concerned], want[name].reshape(400, -1)[~concerned]), name


def test_backward_of_a_frame_that_overflowed(gpu_device):
    """A frame whose keys did not fit has no gradient records, and no room for them: every gradient is zero, nothing is read
    or written past the scratch."""
    scene = scenes.tiny_scene(P=3000, width=160, height=128, sh_degree=1, seed=2)
    s = settings_for(scene, gpu_device)
    inp = pipeline.FrameInputs(s, scene.means3D.to(gpu_device), opacities=scene.opacities.to(gpu_device),
                               shs=scene.shs.to(gpu_device), scales=scene.scales.to(gpu_device),
                               rotations=scene.rotations.to(gpu_device))
    ws = pipeline.Workspace(gpu_device)
    out = pipeline.render(inp, ws=ws)
    image = torch.ones_like(out.image)
    assert pipeline.render_backward(inp, out, ws.buffer, image)["opacities"].any()
    few = out.num_keys // 4
    layout = pipeline.run_stages(inp, out, ws, few, _lib.PIPELINE_FAST)
    out.key_capacity = few
    assert _lib.Header.from_buffer_copy(ws.view(layout, "header", 0, 0, 0).cpu().numpy()).overflow
    grads = pipeline.render_backward(inp, out, ws.buffer, image)
    torch.cuda.synchronize()
    assert all(not g.any() for g in grads.values())
