"""Gradients of Gaussians that cover from one to hundreds of tiles (their key records are added by one lane or by many)
against the oracle."""
import pytest
import torch

from landmarksystem_amd import scenes
from tests.test_gpu_backward import abi_backward, assert_grad_close, cotangents, oracle_backward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,log_scale", [(1, 0.0), (5, -1.0), (64, -1.5), (200, -2.0), (130, 0.0)])
def test_gradients_of_large_splats(gpu_device, P, log_scale):
    scene = scenes.tiny_scene(P=P, width=410, height=300, sh_degree=1, seed=P, log_scale_mean=log_scale)
    g = torch.Generator().manual_seed(P)
    scene.scales = scene.scales * torch.exp(torch.randn(P, 1, generator=g))  # tiles touched: one to all 494
    scene.opacities = scene.opacities * 0.5
    gi, gd, ga = cotangents(scene, P)
    ref, _ = oracle_backward(scene, gi, gd, ga)
    got, _ = abi_backward(scene, gpu_device, gi, gd, ga)
    for name, value in got.items():
        assert_grad_close(value, ref[name], name)
