"""The binning of small frames: slices of less than a workgroup's threads, several lanes per Gaussian, at the edges between
the numbers of lanes and with rectangles on both sides of the queue's threshold, against the classic stages' arrays."""
import numpy as np
import pytest

from landmarksystem_amd import _lib, scenes
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
