"""Keys only for the tiles that a Gaussian's alpha >= 1/255 ellipse reaches (GS355_STAGE_TILE_REACH), against the keys of whole
rectangles: which pairs are left out, and that images and gradients do not change."""
import numpy as np
import pytest
import torch

from landmarksystem_amd import _lib, pipeline, scenes
from oracle import c_oracle as co
from tests.helpers import oracle_frame, oracle_gaussians, settings_for, u32, u64
from tests.test_gpu_parity import crowded_scene

pytestmark = pytest.mark.gpu


def mixed_scene(P=4000, width=431, height=277, seed=1, log_scale=-2.5):
    """Splats of a tile to a whole image, needles among them, opacities from below 1/255 to one, poisoned ones last."""
    scene = scenes.tiny_scene(P=P, width=width, height=height, sh_degree=0, seed=seed)
    g = torch.Generator().manual_seed(seed)
    scene.scales[:] = torch.exp(torch.randn(P, 1, generator=g) * 1.2 + log_scale) * torch.exp(torch.randn(P, 3, generator=g))
    scene.scales[::7, 1:] *= 0.01
    scene.opacities[:] = torch.sigmoid(torch.randn(P, 1, generator=g) * 3.0).reshape(scene.opacities.shape)
    scene.opacities[::11] = 1.0 / 255.0
    nan, inf = float("nan"), float("inf")
    scene.opacities[-1], scene.opacities[-2], scene.opacities[-3], scene.opacities[-4] = nan, -0.5, 0.0, inf
    scene.scales[-5] = torch.tensor([30.0, 1e-6, 1e-6])
    scene.means3D[-6] = torch.tensor([nan, 0.0, 0.0])
    scene.shs[-7] = inf
    return scene


def frame(scene, device, modifiers):
    s = settings_for(scene, device)
    d = scene.to(device)
    inp = pipeline.FrameInputs(s, d.means3D, opacities=d.opacities, shs=d.shs, scales=d.scales, rotations=d.rotations)
    out, ws = pipeline.FrameOutputs(inp), pipeline.Workspace(device)
    n_cap = 8_000_000
    ws.ensure(inp.P, n_cap, inp.width, inp.height)
    ws.buffer.fill_(0xA5)
    lay = pipeline.run_stages(inp, out, ws, n_cap, _lib.PIPELINE_FAST | modifiers)
    torch.cuda.synchronize()
    words = ws.view(lay, "header", inp.P, 0, inp.tiles).cpu().numpy().view(np.uint32)
    n = int(words[2])
    out.key_capacity = n_cap
    return dict(inp=inp, out=out, ws=ws, total=int(words[0]), n=n, visible=int(words[4]),
                keys=u64(ws.view(lay, "sorted_keys", inp.P, n, inp.tiles)),
                values=u32(ws.view(lay, "sorted_values", inp.P, n, inp.tiles)),
                ranges=u32(ws.view(lay, "ranges", inp.P, n, inp.tiles)).astype(np.int64))


def pairs(f):
    return ((f["keys"] >> np.uint64(32)).astype(np.int64) << 32) | f["values"].astype(np.int64)


SCENES = {
    "mixed": mixed_scene, "ragged": lambda: mixed_scene(700, 33, 17, 2), "many": lambda: mixed_scene(40_000, 803, 611, 3, -4.0),
    "serial": lambda: scenes.config3(P=200_000), "crowded": lambda: crowded_scene(3000, width=160, height=96, seed=4),
    "one": lambda: scenes.tiny_scene(P=1, width=40, height=24, sh_degree=0),
    "wide": lambda: scenes.config2(P=20_000, width=4000, height=2400),
}


@pytest.mark.parametrize("name", sorted(SCENES))
@pytest.mark.parametrize("level", [0, _lib.STAGE_TILE_SCATTER_ONE_LEVEL, _lib.STAGE_TILE_SCATTER_TWO_LEVEL])
def test_reached_tiles_only(gpu_device, name, level):
    scene = SCENES[name]()
    full, got = frame(scene, gpu_device, level), frame(scene, gpu_device, level | _lib.STAGE_TILE_REACH)
    assert got["total"] == full["total"] == full["n"] and got["visible"] == full["visible"]
    for plane in ("image", "depth", "alpha", "radii"):
        a, b = getattr(got["out"], plane).cpu().numpy(), getattr(full["out"], plane).cpu().numpy()
        np.testing.assert_array_equal(a, b, err_msg=plane)  # (NaN equals NaN here)
    # what is left is a subset, in the same order, partitioned by its ranges
    p, q = pairs(got), pairs(full)
    keep = np.isin(q, p)
    assert keep.sum() == got["n"] == (got["ranges"][:, 1] - got["ranges"][:, 0]).sum() <= full["n"]
    np.testing.assert_array_equal(q[keep], p)
    np.testing.assert_array_equal(full["keys"][keep], got["keys"])
    tile = (got["keys"] >> np.uint64(32)).astype(np.int64)
    starts = got["ranges"][:, 0][got["ranges"][:, 1] > got["ranges"][:, 0]]
    assert (tile[starts] == np.unique(tile)).all()
    if name in ("mixed", "many", "serial"):
        assert got["n"] < 0.9 * full["n"]
    # and what is left out reaches no pixel of its tile, in double precision from the oracle's splats
    pre = co.preprocess(oracle_frame(scene), oracle_gaussians(scene))
    tiles_x = (scene.camera.width + 15) // 16
    gone = q[~keep][:: max(1, int((~keep).sum()) // 20_000)]
    t, g = gone >> 32, gone & 0xFFFFFFFF
    step = np.arange(16, dtype=np.float64)
    dx = pre["xy"][g, 0].astype(np.float64)[:, None, None] - ((t % tiles_x) * 16)[:, None, None] - step[None, None, :]
    dy = pre["xy"][g, 1].astype(np.float64)[:, None, None] - ((t // tiles_x) * 16)[:, None, None] - step[None, :, None]
    a, b, c, o = (pre["conic_opacity"][g, k].astype(np.float64)[:, None, None] for k in range(4))
    alpha = o * np.exp(-0.5 * (a * dx * dx + c * dy * dy) - b * dx * dy)
    assert not (alpha >= 1.0 / 255.0).any(), float(alpha.max())


@pytest.mark.parametrize("P,log_scale", [(1, 0.0), (63, 0.5), (65, -2.0), (16_384, -3.0), (16_385, -1.5), (131_073, -4.5)])
def test_slices_of_small_frames(gpu_device, P, log_scale):
    """Slices of less than a workgroup's threads, at the edges between the numbers of lanes per Gaussian."""
    scene = scenes.tiny_scene(P=P, width=331, height=203, sh_degree=0, seed=P % 97, log_scale_mean=log_scale)
    full = frame(scene, gpu_device, 0)
    for level in (_lib.STAGE_TILE_SCATTER_ONE_LEVEL, _lib.STAGE_TILE_SCATTER_TWO_LEVEL):
        got = frame(scene, gpu_device, level | _lib.STAGE_TILE_REACH)
        p, q = pairs(got), pairs(full)
        np.testing.assert_array_equal(q[np.isin(q, p)], p)
        assert torch.equal(got["out"].image, full["out"].image)


@pytest.mark.parametrize("make", [lambda: mixed_scene(3000, 331, 203, 5), lambda: scenes.config3(P=300_000),
                                  lambda: scenes.config2(P=300_000, width=640, height=360)],
                         ids=["sums-ahead", "small-splats", "large-splats"])
def test_gradients_do_not_change(gpu_device, make):
    """The records of a region's tiles, summed by one lane, by sixteen (more than 262144 Gaussians) or by a wavefront (up to
    them): sums of the same numbers, in another order where a Gaussian's tiles are dealt out to lanes."""
    scene = make()
    scene.opacities[-8:] = 0.5
    scene.scales[-8:] = 0.1
    scene.means3D[-8:] = scene.means3D[:8].clone()
    scene.shs[-8:] = 0.1
    full, got = frame(scene, gpu_device, 0), frame(scene, gpu_device, _lib.STAGE_TILE_REACH)
    cot = torch.randn(3, scene.camera.height, scene.camera.width, generator=torch.Generator().manual_seed(2)).to(gpu_device)
    cot_d = torch.randn(scene.camera.height, scene.camera.width, generator=torch.Generator().manual_seed(3)).to(gpu_device)
    a = pipeline.render_backward(full["inp"], full["out"], full["ws"].buffer, cot, dL_ddepth=cot_d)
    b = pipeline.render_backward(got["inp"], got["out"], got["ws"].buffer, cot, dL_ddepth=cot_d)
    for name in a:
        x, y = a[name].double(), b[name].double()
        assert torch.isfinite(x).all() and float(x.abs().max()) > 0
        # Sums in two orders.  sum_large_kernel adds n terms in sixteen lanes and those in a tree: of the first scene's 273
        # tiles, 18 terms in a lane and four levels, so at most 21 roundings of 2^-24 in a term's way in either order, 2.5e-6
        # of the terms; the gradients are linear in the sums.  (The others: more tiles, shorter sums.)
        assert float((x - y).norm()) <= 2.5e-6 * float(x.norm()), name
        assert float((x - y).abs().max()) <= 1e-5 * float(x.abs().max()), name


def test_classic_stages_after_it(gpu_device):
    """A workspace whose regions were cut down, then run through the classic stages: their keys are whole rectangles', and the
    backward pass goes by the keys that were blended."""
    scene = mixed_scene(1500, 200, 120, 8)
    scene.opacities[-8:], scene.scales[-8:], scene.shs[-8:] = 0.5, 0.1, 0.1
    scene.means3D[-8:] = scene.means3D[:8].clone()
    full, got = frame(scene, gpu_device, 0), frame(scene, gpu_device, _lib.STAGE_TILE_REACH)
    pipeline.run_stages(got["inp"], got["out"], got["ws"], got["out"].key_capacity, _lib.STAGE_SCAN | _lib.STAGE_DUPLICATE |
                        _lib.STAGE_SORT | _lib.STAGE_RANGES | _lib.STAGE_BLEND)
    assert torch.equal(got["out"].image, full["out"].image)
    cot = torch.randn(3, 120, 200, generator=torch.Generator().manual_seed(2)).to(gpu_device)
    a = pipeline.render_backward(full["inp"], full["out"], full["ws"].buffer, cot)
    b = pipeline.render_backward(got["inp"], got["out"], got["ws"].buffer, cot)
    for name in a:
        assert torch.equal(a[name], b[name]), name


def test_the_scan_remakes_rectangles_only_where_they_were_cut(gpu_device):
    """Whole rectangles are read as the preprocess left them, in the same call or a later one: what has been put in their place
    is still there afterwards.  Parts of them are made whole, once."""
    scene = mixed_scene(5000, 200, 120, 6)
    d = scene.to(gpu_device)
    inp = pipeline.FrameInputs(settings_for(scene, gpu_device), d.means3D, opacities=d.opacities, shs=d.shs, scales=d.scales,
                               rotations=d.rotations)
    out, ws, n_cap = pipeline.FrameOutputs(inp), pipeline.Workspace(gpu_device), 2_000_000
    lay = ws.ensure(inp.P, n_cap, inp.width, inp.height)
    ws.buffer.fill_(0xA5)
    rects = ws.buffer[lay.rects:lay.rects + 8 * inp.P].view(torch.int64)

    def words(*masks):
        for mask in masks:
            pipeline.run_stages(inp, out, ws, n_cap, mask)
        return rects.clone(), ws.view(lay, "offsets", inp.P, 0, inp.tiles).clone()

    whole, offsets = words(_lib.STAGE_PREPROCESS | _lib.STAGE_SCAN)
    mark = 0x0001000100000000  # (one tile, at the corner)
    rects.fill_(mark)
    got = words(_lib.STAGE_SCAN)
    assert bool((got[0] == mark).all()) and torch.equal(got[1], offsets)
    parts, _ = words(_lib.STAGE_PREPROCESS | _lib.STAGE_TILE_REACH)
    assert int((parts != whole).sum()) > 1000
    got = words(_lib.STAGE_SCAN)
    assert torch.equal(got[0], whole) and torch.equal(got[1], offsets)
    rects.fill_(mark)
    got = words(_lib.STAGE_SCAN)
    assert bool((got[0] == mark).all()) and torch.equal(got[1], offsets)
