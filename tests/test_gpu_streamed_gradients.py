"""The preprocess's backward pass reads and writes past the caches in large scenes only: the same gradients to the bit on both sides
of the line, and in small scenes an optimizer's step that finds them in the caches."""
import pytest
import torch

from landmarksystem_amd import GaussianRasterizer, scenes
from landmarksystem_amd.models import GaussianModel
from tests.helpers import settings_for

pytestmark = pytest.mark.gpu

LINE = 1 << 17  # (kStreamedFrom)


@pytest.mark.parametrize("stored,degree,active,depth", [(True, 3, 3, True), (True, 2, 2, False), (True, 3, 0, False), (True, 0, 0, True),
                                                        (False, 3, 3, False), (False, 3, 0, True), (False, 2, 1, False)])
def test_same_gradients_on_both_sides_of_the_line(gpu_device, stored, degree, active, depth):
    scene = scenes.tiny_scene(P=LINE, width=150, height=97, sh_degree=degree, spread=2.0, log_scale_mean=-4.0, seed=degree)
    scene.means3D[LINE - 1, 2] = -100.0  # (behind the camera: the frame is the same without it)
    weights = torch.randn(3, 97, 150, generator=torch.Generator().manual_seed(1)).to(gpu_device)
    grads = []
    for P in (LINE, LINE - 1):
        cut = [t[:P].contiguous().to(gpu_device) for t in (scene.means3D, scene.opacities, scene.shs, scene.scales, scene.rotations)]
        if stored:
            cut = [cut[0], torch.logit(cut[1]), cut[2][:, :1].contiguous(), cut[2][:, 1:].contiguous(), cut[3].log(), cut[4]]
        leaves = [t.requires_grad_(True) for t in cut] + [torch.zeros(P, 3, device=gpu_device, requires_grad=True)]
        r = GaussianRasterizer(settings_for(scene, gpu_device, sh_degree=active))
        if stored:
            xyz, opacity, dc, rest, scales, rotations, screen = leaves
            image, radii, z = r.forward_parameters(xyz, screen, dc, rest, opacity, scales, rotations)
        else:
            xyz, opacity, shs, scales, rotations, screen = leaves
            image, radii, z = r(means3D=xyz, means2D=screen, shs=shs, opacities=opacity, scales=scales, rotations=rotations)
        ((image * weights).sum() + (0.1 * z.sum() if depth else 0.0)).backward()
        assert int((radii[:LINE - 1] > 0).sum()) > LINE // 4 and (P < LINE or int(radii[-1]) == 0)
        grads.append([t.grad[:LINE - 1] for t in leaves])
    assert bool(grads[0][0].any())
    for a, b in zip(*grads):
        assert torch.equal(a, b)


def test_an_optimizer_finds_the_gradients_of_a_small_scene_in_the_caches(gpu_device):
    """Adam's step behind a pass over 100k Gaussians, against the same step behind a pass whose gradients and parameters were read
    once more by ordinary accesses (1.23 times as long where the pass streams them)."""
    scene = scenes.config2(P=100_003, width=800, height=533)
    model = GaussianModel.from_activated(scene.means3D, scene.scales, scene.rotations, scene.opacities, scene.shs[:, :9].contiguous(),
                                         sh_degree=2).to(gpu_device).train()
    params = [model._xyz, model._features_dc, model._features_rest, model._scaling, model._rotation, model._opacity]
    for p in params:
        p.requires_grad_(True)
    adam = torch.optim.Adam(params, lr=1e-12, fused=True)
    times = {False: [], True: []}
    for k in range(80):
        for p in params:
            p.grad = None
        model(scene.camera).sum().backward()
        touched = k % 2 == 1
        if touched:
            for p in params:
                p.grad.mul_(1.0)
                p.data.mul_(1.0)
        start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda._sleep(400_000)  # (the host is ahead when the step begins)
        start.record()
        adam.step()
        stop.record()
        torch.cuda.synchronize()
        times[touched].append(1e3 * start.elapsed_time(stop))
    plain, touched = (sorted(times[t][10:])[15] for t in (False, True))
    print("Adam's step: %.1f us behind the pass, %.1f us with everything touched" % (plain, touched))
    assert plain < 1.12 * touched
