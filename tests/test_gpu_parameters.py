"""Frames and gradients taken from GaussianModel's stored parameters inside the kernels, against the same frame over the
activated tensors (whose own parity with the oracle the other tests hold)."""
import ctypes as C

import pytest
import torch

from landmarksystem_amd import GaussianRasterizer, _lib, pipeline, scenes
from landmarksystem_amd.models import GaussianModel
from tests.helpers import settings_for
from tests.test_gpu_backward import assert_grad_close

pytestmark = pytest.mark.gpu


# counts around the staging's wavefront and workgroup, and rows of 45 floats whose total is no multiple of four
@pytest.mark.parametrize("P,degree,active", [(1, 3, 3), (2, 3, 3), (63, 0, 0), (65, 1, 1), (257, 2, 2), (258, 3, 1),
                                             (1003, 3, 3), (30_001, 3, 3), (4096, 3, 0)])
def test_stored_parameters_render_as_activated_ones(gpu_device, P, degree, active):
    scene = scenes.tiny_scene(P=P, width=150, height=97, sh_degree=degree, log_scale_mean=-2.5)
    g = torch.Generator().manual_seed(P)
    rot = scene.rotations * (0.2 + 2.0 * torch.rand(P, 1, generator=g))
    if P > 2:
        rot[1] = 0.0  # (the normalisation's floor)
    model = GaussianModel.from_activated(scene.means3D, scene.scales, rot, scene.opacities, scene.shs, sh_degree=degree)
    model = model.to(gpu_device).train()
    leaves = dict(means3D=model._xyz, shs=model._features_dc, features_rest=model._features_rest,
                  opacities=model._opacity, scales=model._scaling, rotations=model._rotation)
    for p in leaves.values():
        p.requires_grad_(True)
    model.active_sh_degree = active
    r = GaussianRasterizer(settings_for(scene, gpu_device, sh_degree=active))
    weights = torch.randn(3, 97, 150, generator=g).to(gpu_device)
    results = []
    for stored in (True, False):
        means2D = torch.zeros(P, 3, device=gpu_device, requires_grad=True)
        for p in leaves.values():
            p.grad = None
        if stored:
            image, radii, depth = r.forward_parameters(model._xyz, means2D, model._features_dc, model._features_rest,
                                                       model._opacity, model._scaling, model._rotation)
        else:
            image, radii, depth = r(means3D=model.get_xyz, means2D=means2D, shs=model.get_features,
                                    opacities=model.get_opacity, scales=model.get_scaling, rotations=model.get_rotation)
        (image * weights + depth * 0.1).sum().backward()
        results.append((image.detach(), radii, depth.detach(),
                        {n: p.grad.cpu().numpy() for n, p in dict(leaves, means2D=means2D).items()}))
    (image_s, radii_s, depth_s, grads_s), (image_a, radii_a, depth_a, grads_a) = results
    assert torch.equal(radii_s, radii_a) and torch.equal(image_s, image_a) and torch.equal(depth_s, depth_a)
    for name, want in grads_a.items():
        assert grads_s[name].shape == want.shape
        if want.size:
            assert_grad_close(grads_s[name], want, name)


def test_training_model_takes_the_stored_parameters(gpu_device):
    scene = scenes.tiny_scene(P=500, width=80, height=64, sh_degree=2)
    model = GaussianModel.from_activated(scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs,
                                         sh_degree=2).to(gpu_device).train()
    for p in model.parameters():
        p.requires_grad_(True)
    assert model._renders_parameters()
    image = model(scene.camera)
    image.sum().backward()
    assert model.viewspace_points.grad.shape == model._xyz.shape and model.radii.shape == (500,)
    model.compute_cov3D_python = True  # (the activated tensors again)
    assert not model._renders_parameters()
    assert torch.allclose(model(scene.camera), image, atol=1e-4)


def test_parameters_replaced_before_the_backward_pass(gpu_device):
    """Densification between the passes: the backward pass refuses a scene of another size (the workspace and the radii are
    those of the forward pass)."""
    scene = scenes.tiny_scene(P=500, width=80, height=64, sh_degree=2)
    model = GaussianModel.from_activated(scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs,
                                         sh_degree=2).to(gpu_device).train()
    for p in model.parameters():
        p.requires_grad_(True)
    image = model(scene.camera)
    for p in (model._xyz, model._features_dc, model._features_rest, model._opacity, model._scaling, model._rotation):
        p.data = torch.cat([p.data, p.data])
    with pytest.raises(RuntimeError, match="number of Gaussians"):
        image.sum().backward()
    torch.cuda.synchronize()


@pytest.mark.parametrize("A,columns", [(1, 6), (63, 3), (64, 6), (65, 4), (1023, 6), (100_001, 6)])
def test_anchor_filter_over_stored_parameters(gpu_device, A, columns):
    """gs355_anchor_filter_parameters against gs355_anchor_filter over the activated tensors: the same anchors, sizes down to
    a pixel's (where the last bit of a scale decides) and quaternions down to zero among them."""
    scene = scenes.tiny_scene(P=A, width=150, height=97, sh_degree=0)
    g = torch.Generator().manual_seed(A)
    anchors = (scene.means3D * 2.0).to(gpu_device)
    scaling = (torch.randn(A, columns, generator=g) * 2.0 - 4.0).to(gpu_device)
    rotation = (torch.randn(A, 4, generator=g) * torch.exp(torch.randn(A, 1, generator=g) * 4.0)).to(gpu_device)
    if A > 2:
        rotation[1], rotation[2] = 0.0, 1e-20
    s = settings_for(scene, gpu_device)
    stored, none = pipeline.anchor_filter(s, anchors, scaling, rotation, stored=True)
    want, _ = pipeline.anchor_filter(s, anchors, torch.exp(scaling), torch.nn.functional.normalize(rotation))
    assert none is None and torch.equal(stored, want)
    assert A < 60 or 0 < int(want.sum()) < A


@pytest.mark.parametrize("stored", [False, True])
def test_frame_call_reports_an_overflow_and_is_repeated(gpu_device, stored):
    """gs355_render_frame itself: too small a capacity comes back with the exact number of keys in the header, the same
    call with that capacity renders the frame."""
    scene = scenes.tiny_scene(P=3000, width=160, height=128, sh_degree=2, seed=2)
    model = GaussianModel.from_activated(scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs,
                                         sh_degree=2).to(gpu_device)
    s = settings_for(scene, gpu_device)
    if stored:
        inp = pipeline.FrameInputs(s, model._xyz, opacities=model._opacity, shs=model._features_dc, scales=model._scaling,
                                   rotations=model._rotation, features_rest=model._features_rest)
    else:
        inp = pipeline.FrameInputs(s, model.get_xyz, opacities=model.get_opacity, shs=model.get_features,
                                   scales=model.get_scaling, rotations=model.get_rotation)
    want = pipeline.render(inp, ws=pipeline.Workspace(gpu_device))
    ws, out = pipeline.Workspace(gpu_device), pipeline.FrameOutputs(inp)
    out.c.header_copy = ws.header_host.data_ptr()

    def call(n_cap):
        ws.ensure(inp.P, n_cap, inp.width, inp.height)
        _lib.check(_lib.load().gs355_render_frame(
            C.byref(inp.frame), C.byref(inp.gaussians), int(stored), pipeline._ptr(inp.features_rest), ws.buffer.data_ptr(),
            ws.buffer.numel(), n_cap, C.byref(out.c), _lib.PIPELINE_FAST, pipeline._raw_stream(gpu_device)))
        h = ws.header
        return h.ready, h.overflow, h.num_keys_total, h.num_visible

    assert call(want.num_keys - 1) == (1, 1, want.num_keys, want.num_visible)
    assert call(want.num_keys) == (1, 0, want.num_keys, want.num_visible)
    for a, b in ((out.image, want.image), (out.depth, want.depth), (out.alpha, want.alpha), (out.radii, want.radii)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("P", [1, 255, 257, 5000])
def test_coefficient_blocks_off_their_boundary(gpu_device, P):
    """Blocks of 16 coefficients at 16-byte boundaries travel through LDS, others are read by their own lanes, in a kernel
    without that room: the same sums in the same order."""
    scene = scenes.tiny_scene(P=P, width=331, height=203, sh_degree=3, seed=P % 97)
    settings = settings_for(scene, gpu_device)
    d = scene.to(gpu_device)
    room = torch.empty(P * 48 + 4, device=gpu_device)
    outs = []
    for first in (0, 1):
        shs = room[first:first + P * 48].view(P, 16, 3)
        shs.copy_(d.shs)
        assert shs.data_ptr() % 16 == 4 * first
        inp = pipeline.FrameInputs(settings, d.means3D, opacities=d.opacities, shs=shs, scales=d.scales, rotations=d.rotations)
        out = pipeline.render(inp, ws=pipeline.Workspace(gpu_device))
        outs.append((out.image.clone(), out.depth.clone(), out.radii.clone()))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
