"""The binning of small frames: slices of less than a workgroup's threads, several lanes per Gaussian, at the edges between
the numbers of lanes and with rectangles on both sides of the queue's threshold, against the classic stages' arrays."""
import numpy as np
import pytest
import torch

from landmarksystem_amd import _lib, pipeline, scenes
from tests.helpers import settings_for
from tests.test_gpu_parity import crowded_scene, run_all_stages, run_fast_path

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,log_scale", [(1, 0.0), (63, 0.5), (65, -2.0), (16_384, -3.0), (16_385, -1.5), (32_769, -3.0),
                                         (65_537, -4.0), (131_072, -4.0), (131_073, -4.5)])
def test_slices_of_small_frames(gpu_device, P, log_scale):
    scene = scenes.tiny_scene(P=P, width=331, height=203, sh_degree=0, seed=P % 97, log_scale_mean=log_scale)
    want = run_all_stages(scene, gpu_device)
    for two_level in (False, True):
        got = run_fast_path(scene, gpu_device, two_level=two_level)
        for name in ("ranges", "sorted_keys", "sorted_values"):
            np.testing.assert_array_equal(got[name], want[name], err_msg="%d %s" % (P, name))


def one_depth():
    """600 of 800 pairs of every bucket at one depth: more than a bin of the counting sort takes."""
    scene = crowded_scene(800)
    scene.means3D[:600] = scene.means3D[0].clone()
    return scene


@pytest.mark.parametrize("make,skip", [
    (lambda: scenes.config2(P=100_000), 0), (lambda: scenes.config3(P=300_000), 0),
    (lambda: crowded_scene(3000, width=1000, height=700, duplicates=100), 0),
    (lambda: crowded_scene(3000, width=1000, height=700, duplicates=100), sum(_lib.STAGE_TILESORT_SKIP)),
    (lambda: crowded_scene(8000, width=32, height=32, duplicates=500), 0),
    (lambda: crowded_scene(12_000, width=32, height=32, duplicates=700), 0), (one_depth, 0)],
    ids=["large-splats", "small-splats", "lists", "lists-left-out", "largest", "beyond-LDS", "one-depth"])
def test_sorted_values_without_their_keys(gpu_device, make, skip):
    scene = make()
    want = run_fast_path(scene, gpu_device, modifiers=skip)
    got = run_fast_path(scene, gpu_device, modifiers=skip | _lib.STAGE_TILESORT_VALUES)
    for name in ("ranges", "sorted_values", "image", "depth", "alpha"):
        np.testing.assert_array_equal(got[name], want[name], err_msg=name)


@pytest.mark.parametrize("width,height,P,log_scale", [
    (16, 16, 70, 0.0), (48, 16, 12_000, 0.5), (16 * 63, 16, 3000, -2.0), (16 * 64, 16, 3000, -2.0), (16 * 65, 16, 3000, -2.0), (1000, 700, 9000, -2.5),
    (16 * 1023, 16, 20_000, -2.5), (4096, 2304, 40_000, -5.0), (16 * 360, 1600, 40_000, -5.0)])
@pytest.mark.parametrize("levels", [0, _lib.STAGE_TILE_SCATTER_ONE_LEVEL, _lib.STAGE_TILE_SCATTER_TWO_LEVEL])
def test_layout_made_by_the_scatter(gpu_device, width, height, P, log_scale, levels):
    """Tile count and scatter in one call, where the scatter makes the layout, against one call each: at the edges of the
    layout's blocks of 64 tiles and of a workgroup's sixteen of them, up to the 36000 tiles of the LDS counters; with buckets
    beyond 10240 pairs; and for a capacity one key short."""
    scene = scenes.tiny_scene(P=P, width=width, height=height, sh_degree=0, seed=3, log_scale_mean=log_scale)
    inp = pipeline.FrameInputs(settings_for(scene, gpu_device), scene.means3D.to(gpu_device), shs=scene.shs.to(gpu_device),
                               opacities=scene.opacities.to(gpu_device), scales=scene.scales.to(gpu_device),
                               rotations=scene.rotations.to(gpu_device))
    tiles = inp.tiles

    def frame(joint, n_cap):
        out, ws = pipeline.FrameOutputs(inp), pipeline.Workspace(gpu_device)
        lay = ws.ensure(P, n_cap, width, height)
        ws.buffer.fill_(0xA5)
        if joint:
            masks = (_lib.STAGE_PREPROCESS, _lib.STAGE_TILE_COUNT | _lib.STAGE_TILE_SCATTER | levels)
        else:
            masks = (_lib.STAGE_PREPROCESS, _lib.STAGE_TILE_COUNT, _lib.STAGE_TILE_SCATTER | levels)
        for mask in masks + (_lib.STAGE_TILESORT,):
            pipeline.run_stages(inp, out, ws, n_cap, mask)
        torch.cuda.synchronize()
        raw = ws.buffer.cpu().numpy()
        header = raw[lay.header:lay.header + 48].view(np.uint32)  # (up to sort_beyond_count)
        lists = raw[lay.tile_lists:lay.tile_lists + 4 * (8 + 4 * tiles)].view(np.uint32)
        got = {"header": header}
        if header[3] == 0:
            n = int(header[2])
            got["ranges"] = raw[lay.ranges:lay.ranges + 8 * tiles].view(np.uint32)
            got["keys"] = ws.view(lay, "sorted_keys", P, n, tiles).cpu().numpy()
            got["values"] = ws.view(lay, "sorted_values", P, n, tiles).cpu().numpy()
            got["counts"] = lists[:3]
            n = got["ranges"].reshape(tiles, 2)
            beyond = (n[:, 1] - n[:, 0] > 10240).sum() if tiles <= 36000 else 0xFFFFFFFF  # (not counted)
            assert header[11] == beyond and (P != 12_000 or beyond == 3)
            for c in range(3):
                got["list %d" % c] = np.sort(lists[8 + c * tiles:][:lists[c]])
        return got

    total = int(frame(False, 1 << 25)["header"][0])
    assert 0 < total < 1 << 25
    for n_cap in (total, total - 1):
        want, got = frame(False, n_cap), frame(True, n_cap)
        assert want["header"][3] == (n_cap < total) and want.keys() == got.keys()
        for name in want:
            np.testing.assert_array_equal(got[name], want[name], err_msg=name)


@pytest.mark.parametrize("width,height,P,log_scale", [
    (16, 16, 70, 0.0), (16 * 65, 16, 3000, -2.0), (1000, 700, 9000, -2.5), (16 * 1023, 16, 20_000, -2.5), (16 * 360, 1600, 40_000, -5.0)])
def test_scattered_again_in_two_levels(gpu_device, width, height, P, log_scale):
    """Tile count and scatter in one level in one call, then the scatter by itself in two: the work list of its second level (bins of
    16 tiles, as many as 2250) is there, and the pairs end where they did."""
    scene = scenes.tiny_scene(P=P, width=width, height=height, sh_degree=0, seed=4, log_scale_mean=log_scale)
    inp = pipeline.FrameInputs(settings_for(scene, gpu_device), scene.means3D.to(gpu_device), shs=scene.shs.to(gpu_device),
                               opacities=scene.opacities.to(gpu_device), scales=scene.scales.to(gpu_device),
                               rotations=scene.rotations.to(gpu_device))
    out, ws, tiles, n_cap = pipeline.FrameOutputs(inp), pipeline.Workspace(gpu_device), inp.tiles, 1 << 24
    lay = ws.ensure(P, n_cap, width, height)
    ws.buffer.fill_(0x0)
    run = lambda mask: pipeline.run_stages(inp, out, ws, n_cap, mask)  # noqa: E731
    run(_lib.STAGE_PREPROCESS)
    run(_lib.STAGE_TILE_COUNT | _lib.STAGE_TILE_SCATTER | _lib.STAGE_TILE_SCATTER_ONE_LEVEL)
    at = lay.tile_base + 4 * (2 * tiles + 2 * ((tiles + 63) // 64))
    bins = (tiles + 15) // 16
    chunks = ws.buffer[at:at + 4 * (bins + 1)].view(torch.int32).cpu().numpy()
    ranges = ws.view(lay, "ranges", P, 0, tiles).cpu().numpy()
    n = np.pad(ranges[:, 1] - ranges[:, 0], (0, 16 * bins - tiles)).reshape(bins, 16).sum(1)
    np.testing.assert_array_equal(chunks, np.concatenate([[0], np.cumsum((n + 2047) // 2048)]))
    assert n.sum() > 0
    run(_lib.STAGE_TILESORT)
    want = [ws.view(lay, name, P, int(n.sum()), tiles).clone() for name in ("sorted_keys", "sorted_values")]
    run(_lib.STAGE_TILE_SCATTER | _lib.STAGE_TILE_SCATTER_TWO_LEVEL)
    run(_lib.STAGE_TILESORT)
    for a, name in zip(want, ("sorted_keys", "sorted_values")):
        assert torch.equal(ws.view(lay, name, P, int(n.sum()), tiles), a), name


@pytest.mark.parametrize("width,height,P,log_scale", [
    (256, 256, 900, -1.0), (16 * 257, 16, 3000, -1.5), (512, 256, 2000, -2.0), (513, 256, 2000, -2.0), (1000, 700, 9000, -2.5),
    (1000, 700, 9000, -5.0), (16 * 360, 1600, 4000, -2.5), (16 * 360, 1600, 30_000, -5.0), (16 * 361, 1600, 4000, -2.5)])
def test_tiles_in_the_order_of_their_lists(gpu_device, width, height, P, log_scale):
    """The tile sort's order of the tiles: each of them once, with its range, no later than a list of more than 1/16 less; made
    for 257 to 36000 tiles of 128 pairs or more on average; the same image with and without it; and forgotten when a new frame's
    header is written."""
    scene = scenes.tiny_scene(P=P, width=width, height=height, sh_degree=0, seed=5, log_scale_mean=log_scale)
    inp = pipeline.FrameInputs(settings_for(scene, gpu_device), scene.means3D.to(gpu_device), shs=scene.shs.to(gpu_device),
                               opacities=scene.opacities.to(gpu_device), scales=scene.scales.to(gpu_device),
                               rotations=scene.rotations.to(gpu_device))
    out, ws, tiles, n_cap = pipeline.FrameOutputs(inp), pipeline.Workspace(gpu_device), inp.tiles, 1 << 24
    lay = ws.ensure(P, n_cap, width, height)
    ws.buffer.fill_(0xA5)
    run = lambda mask: pipeline.run_stages(inp, out, ws, n_cap, mask)  # noqa: E731
    word = lambda: ws.buffer[lay.header + 40:lay.header + 44].view(torch.int32)  # noqa: E731
    run(_lib.STAGE_PREPROCESS)
    run(_lib.STAGE_TILE_COUNT | _lib.STAGE_TILE_SCATTER)
    assert int(word()) == 0
    run(_lib.STAGE_TILESORT | _lib.STAGE_BLEND)
    pairs = int(ws.view(lay, "header", P, 0, tiles)[1].item()) & 0xFFFFFFFF
    assert pairs > 0 and (pairs >= 128 * tiles) == (log_scale > -5.0)
    made = 257 <= tiles <= 36000 and log_scale > -5.0
    assert int(word()) == made
    image = out.image.clone()
    if made:
        at = lay.tile_lists + 4 * (8 + 4 * tiles)
        order = ws.buffer[at:at + 16 * tiles].view(torch.int32).view(tiles, 4).cpu().numpy()
        ranges = ws.view(lay, "ranges", P, 0, tiles).cpu().numpy()
        assert (np.sort(order[:, 0]) == np.arange(tiles)).all()
        np.testing.assert_array_equal(order[:, 1:3], ranges[order[:, 0]])
        n = (order[:, 2] - order[:, 1]).astype(np.int64)
        assert n.max() > 0 and (np.minimum.accumulate(n) * 17 >= n * 16).all()
        word().zero_()
        out.image.zero_()
        run(_lib.STAGE_BLEND)
        assert torch.equal(out.image, image)
        word().fill_(1)
    run(_lib.STAGE_TILE_COUNT)
    assert int(word()) == 0
    word().fill_(1)
    run(_lib.STAGE_SCAN)
    assert int(word()) == 0


@pytest.mark.parametrize("P,duplicates", [(1, 0), (2, 1), (63, 0), (64, 30), (65, 0), (200, 100), (255, 0), (256, 128), (257, 0)])
@pytest.mark.parametrize("one_depth", [False, True])
def test_buckets_that_a_wavefront_sorts(gpu_device, P, duplicates, one_depth):
    """Every Gaussian in each of 625 tiles: buckets of up to 256 pairs, and one more, with equal depths among them or nothing else."""
    scene = crowded_scene(P, width=400, height=400, duplicates=duplicates)
    if one_depth:
        scene.means3D[:] = scene.means3D[0].clone()
    want = run_all_stages(scene, gpu_device)
    for modifiers in (0, _lib.STAGE_TILESORT_VALUES):
        got = run_fast_path(scene, gpu_device, modifiers=modifiers)
        for name in ("ranges", "sorted_keys", "sorted_values")[::2 if modifiers else 1]:
            np.testing.assert_array_equal(got[name], want[name], err_msg="%d %s" % (P, name))


@pytest.mark.parametrize("P,equal", [(10240, 0), (10241, 0), (10241, 10241), (16384, 100), (16385, 100), (20500, 3000), (31000, 100), (24000, 12000), (31000, 31000)])
@pytest.mark.parametrize("side", [32, 400])
def test_buckets_beyond_the_lds(gpu_device, P, equal, side):
    """Every Gaussian in each of 4 or 625 tiles: one piece, several, equal depths among them, and more of those in one bin than
    the LDS sorter holds (alone, and between other bins)."""
    scene = crowded_scene(P, width=side, height=side)
    if equal:
        scene.means3D[::P // equal][:equal] = scene.means3D[0].clone()
    want = run_all_stages(scene, gpu_device)
    assert (want["ranges"][:, 1] - want["ranges"][:, 0]).max() == P
    for modifiers in (0, _lib.STAGE_TILESORT_VALUES):
        got = run_fast_path(scene, gpu_device, modifiers=modifiers)
        for name in ("ranges", "sorted_keys", "sorted_values")[::2 if modifiers else 1]:
            np.testing.assert_array_equal(got[name], want[name], err_msg="%d %s" % (P, name))
    # their launch is not left out where the frames before held only such buckets
    scene.opacities[:] = 0.05
    inputs = pipeline.FrameInputs(settings_for(scene, gpu_device), scene.means3D.to(gpu_device),
                                  opacities=scene.opacities.to(gpu_device), shs=scene.shs.to(gpu_device),
                                  scales=scene.scales.to(gpu_device), rotations=scene.rotations.to(gpu_device))
    ws = pipeline.Workspace(gpu_device)
    for _ in range(6):
        pipeline.render(inputs, ws=ws)
    header = ws.header
    assert P < 12_000 or side > 32 or header.sort_beyond_count > 0
    assert (ws.sort_class_idle[2] == 0) == (header.sort_class_count[2] + header.sort_beyond_count > 0)
    assert ws.sort_mispredictions == 0


@pytest.mark.parametrize("P", [(1 << 24) - 1, 1 << 24])
def test_buckets_of_all_that_a_float_counts(gpu_device, P):
    """One tile of 2^24 pairs, which radix passes through global memory sort, and one of a pair fewer, which is the largest that
    is split by depth: ordered by depth, and by index where depths are equal."""
    scene = crowded_scene(P, width=16, height=16)
    inp = pipeline.FrameInputs(settings_for(scene, gpu_device), *(t.to(gpu_device) for t in (scene.means3D, scene.opacities, scene.shs)),
                               scales=scene.scales.to(gpu_device), rotations=scene.rotations.to(gpu_device))
    out, ws = pipeline.FrameOutputs(inp), pipeline.Workspace(gpu_device)
    for mask in (_lib.STAGE_PREPROCESS, _lib.STAGE_TILE_COUNT | _lib.STAGE_TILE_SCATTER, _lib.STAGE_TILESORT):
        lay = pipeline.run_stages(inp, out, ws, P, mask)
    assert ws.view(lay, "ranges", P, P, 1).tolist() == [[0, P]]
    depth, index = ws.view(lay, "sorted_keys", P, P, 1), ws.view(lay, "sorted_values", P, P, 1).long()
    assert bool((depth >> 32 == 0).all())
    own = ws.buffer[lay.depth_bits:lay.depth_bits + 4 * P].view(torch.int32)
    assert torch.equal(own[index].long(), depth)
    step = depth.diff()
    assert bool(((step > 0) | ((step == 0) & (index.diff() > 0))).all())


@pytest.mark.parametrize("P,pairs", [(8500, (3, 6)), (13_000, (6, 12)), (24_000, (12, 18))])
@pytest.mark.parametrize("form", ["shs", "colours", "count"])
def test_frames_between_the_scatters_thresholds(gpu_device, monkeypatch, form, P, pairs):
    """3 to 6, 6 to 12 and more Mi pairs: the first frame of a workspace scatters in one level, the second as its pairs and the
    Gaussians' form say, and the images are the same."""
    scene = crowded_scene(P, width=400, height=400)
    scene.opacities[:] = 0.05
    scene.scales[:] = scene.scales.clamp(min=1.5)
    at = lambda x: x.to(gpu_device)
    colour = dict(shs=at(scene.shs)) if form == "shs" else dict(colors_precomp=at(scene.shs[:, 0].contiguous()).abs())
    if form == "count":
        colour["count"] = torch.tensor([scene.P], dtype=torch.int32, device=gpu_device)
    inputs = pipeline.FrameInputs(settings_for(scene, gpu_device), at(scene.means3D), opacities=at(scene.opacities),
                                  scales=at(scene.scales), rotations=at(scene.rotations), **colour)
    ws, named = pipeline.Workspace(gpu_device), []
    render_frame = _lib.load().gs355_render_frame

    def watched(*args):
        named.append(args[-2] & (_lib.STAGE_TILE_SCATTER_ONE_LEVEL | _lib.STAGE_TILE_SCATTER_TWO_LEVEL))
        return render_frame(*args)

    monkeypatch.setattr(_lib.load(), "gs355_render_frame", watched)
    first = pipeline.render(inputs, ws=ws)
    assert pairs[0] << 20 <= ws.last_num_pairs < pairs[1] << 20, ws.last_num_pairs
    assert set(named) == {_lib.STAGE_TILE_SCATTER_ONE_LEVEL}
    two = pairs[0] >= (12 if form == "count" else 6)
    for _ in range(2):
        named.clear()
        again = pipeline.render(inputs, ws=ws)
        assert named == [_lib.STAGE_TILE_SCATTER_TWO_LEVEL if two else _lib.STAGE_TILE_SCATTER_ONE_LEVEL]
        for name in ("image", "depth", "alpha"):
            assert torch.equal(getattr(again, name), getattr(first, name)), name
