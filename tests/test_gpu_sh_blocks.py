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
    lay = pipeline.run_stages(inp, out, ws, 1 << 10, _lib.STAGE_PREPROCESS)
    records = ws.view(lay, "records", inp.P, 0, inp.tiles)[out.radii > 0].clone()
    return records.view(torch.int32), out.radii.clone()


# Rows of 9, 12, 24, 27, 45 and 48 floats, whose last one ends on every remainder of a 16-byte chunk, in scenes of as many Gaussians
# as it takes (four coefficients: 2^19, nine: 2^17); one survivor, all, and workgroups of which few survive.
@pytest.mark.parametrize("stored", [False, True])
@pytest.mark.parametrize("degree,P,active,spread", [
    (1, 1 << 19, 1, 1.0), (1, (1 << 19) + 1, 1, 6.0), (1, (1 << 19) + 2, 0, 3.0), (1, (1 << 19) + 63, 1, 1.0),
    (2, 1 << 17, 2, 1.0), (2, (1 << 17) + 1, 1, 6.0), (2, (1 << 17) + 2, 0, 3.0), (2, (1 << 17) + 67, 2, 1.0),
    (3, 1, 3, 0.1), (3, 2, 3, 0.1), (3, 3, 1, 0.1), (3, 63, 2, 1.0), (3, 258, 3, 6.0), (3, 5000, 0, 3.0)])
def test_blocks_through_lds_give_the_same_colours(gpu_device, stored, degree, P, active, spread):
    scene = scenes.tiny_scene(P=P, width=150, height=97, sh_degree=degree, spread=spread, seed=P)
    scales, opacities = scene.scales.to(gpu_device), scene.opacities.to(gpu_device)
    shs, rest = scene.shs.to(gpu_device), None
    if stored:
        scales, opacities = scales.log(), torch.logit(opacities)
        shs, rest = shs[:, :1].contiguous(), shs[:, 1:].contiguous()
    got = _frame(scene, gpu_device, shs, rest, scales, scene.rotations.to(gpu_device), opacities, active)
    want = _frame(scene, gpu_device, shs if stored else _off_boundary(shs), _off_boundary(rest) if stored else None, scales,
                  scene.rotations.to(gpu_device), opacities, active)
    assert int((want[1] > 0).sum()) > 0
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("degree", [0, 1, 2, 3])
@pytest.mark.parametrize("spread", [1.0, 6.0, 40.0])  # nearly all survive, a third, few enough that a wavefront's rows have no room
def test_records_that_leave_by_the_line(gpu_device, degree, spread):
    """The same Gaussians in a scene of 2^19 and more, and one by one over the edge of it: the same records."""
    P = (1 << 19) + 70
    scene = scenes.tiny_scene(P=P, width=150, height=97, sh_degree=degree, spread=spread, seed=degree)
    records = []
    for first, n in ((0, P), (0, (1 << 19) - 1), (100, P - 100)):
        d = [t[first:first + n].contiguous().to(gpu_device) for t in (scene.means3D, scene.opacities, scene.shs, scene.scales, scene.rotations)]
        inp = pipeline.FrameInputs(settings_for(scene, gpu_device), d[0], opacities=d[1], shs=d[2], scales=d[3], rotations=d[4])
        out, ws = pipeline.FrameOutputs(inp), pipeline.Workspace(gpu_device)
        lay = pipeline.run_stages(inp, out, ws, 1 << 10, _lib.STAGE_PREPROCESS)
        rows = ws.view(lay, "records", n, 0, inp.tiles).view(torch.int32)
        keep = (torch.arange(n, device=gpu_device) + first < (1 << 19) - 1) & (torch.arange(n, device=gpu_device) + first >= 100) & (out.radii > 0)
        records.append(rows[keep].clone())
    assert records[0].shape[0] > 10
    assert torch.equal(records[0], records[1]) and torch.equal(records[0], records[2])


@pytest.mark.parametrize("degree,spread", [(0, 1.0), (3, 6.0)])
def test_records_that_are_streamed(gpu_device, degree, spread):
    """The same Gaussians in a scene of 2^21 and in one of one fewer: the same records."""
    P = 1 << 21
    scene = scenes.tiny_scene(P=P, width=150, height=97, sh_degree=degree, spread=spread, seed=degree)
    records = []
    for n in (P, P - 1):
        d = [t[:n].contiguous().to(gpu_device) for t in (scene.means3D, scene.opacities, scene.shs, scene.scales, scene.rotations)]
        inp = pipeline.FrameInputs(settings_for(scene, gpu_device), d[0], opacities=d[1], shs=d[2], scales=d[3], rotations=d[4])
        out, ws = pipeline.FrameOutputs(inp), pipeline.Workspace(gpu_device)
        lay = pipeline.run_stages(inp, out, ws, 1 << 10, _lib.STAGE_PREPROCESS)
        rows = ws.view(lay, "records", n, 0, inp.tiles).view(torch.int32)
        records.append(rows[:P - 1][out.radii[:P - 1] > 0].clone())
    assert records[0].shape[0] > 1000 and torch.equal(records[0], records[1])
