"""Colours from SH blocks of 4, 9 and 16 coefficients, which travel through LDS, against the same blocks read by a lane each (as
they are where their array does not start on a 16-byte boundary): the same values to the bit."""
import pytest
import torch

from landmarksystem_amd import _lib, pipeline, scenes
from tests.helpers import settings_for

pytestmark = pytest.mark.gpu


def _off_boundary(t):
    """The same values one float behind a 16-byte boundary."""
    room = torch.empty(t.numel() + 1, device=t.device)
    room[1:] = t.reshape(-1)
    return room[1:].view(t.shape)


def _frame(scene, device, shs, rest, scales, rotations, opacities, active):
    inp = pipeline.FrameInputs(settings_for(scene, device, sh_degree=active), scene.means3D.to(device), opacities=opacities, shs=shs,
                               scales=scales, rotations=rotations, features_rest=rest)
    out, ws = pipeline.FrameOutputs(inp), pipeline.Workspace(device)
    lay = pipeline.run_stages(inp, out, ws, 1 << 20, _lib.PIPELINE_FAST)
    records = ws.view(lay, "records", inp.P, 0, inp.tiles)[out.radii > 0].clone()
    return records.view(torch.int32), out.image.clone(), out.radii.clone()


# rows of 9, 12, 24, 27, 45 and 48 floats, whose last one ends on every remainder of a 16-byte chunk; one survivor, all, and a
# workgroup of which few survive
@pytest.mark.parametrize("stored", [False, True])
@pytest.mark.parametrize("degree", [1, 2, 3])
@pytest.mark.parametrize("P,active,spread", [(1, 1, 0.1), (2, 1, 0.1), (3, 0, 0.1), (63, 1, 1.0), (258, 1, 6.0), (1027, 1, 1.0), (5000, 1, 3.0)])
def test_blocks_through_lds_give_the_same_colours(gpu_device, stored, degree, P, active, spread):
    scene = scenes.tiny_scene(P=P, width=150, height=97, sh_degree=degree, spread=spread, seed=P)
    scales, opacities = scene.scales.to(gpu_device), scene.opacities.to(gpu_device)
    shs, rest = scene.shs.to(gpu_device), None
    if stored:
        scales, opacities = scales.log(), torch.logit(opacities)
        shs, rest = shs[:, :1].contiguous(), shs[:, 1:].contiguous()
    for sh_degree in (active, degree):
        got = _frame(scene, gpu_device, shs, rest, scales, scene.rotations.to(gpu_device), opacities, sh_degree)
        want = _frame(scene, gpu_device, shs if stored else _off_boundary(shs), _off_boundary(rest) if stored else None, scales,
                      scene.rotations.to(gpu_device), opacities, sh_degree)
        assert int((want[2] > 0).sum()) > 0
        for a, b in zip(got, want):
            assert torch.equal(a, b)
