"""The raw backward's inputs: what it converts stays alive until its launches, and what it cannot use is refused
before any of them."""

from __future__ import annotations

import pytest
import torch

from gswarp_amd import _lib, _rasterizer, configs
from helpers import raster_inputs

pytestmark = pytest.mark.gpu


def _call(device, side: int = 8, count: int = 40):
    """(inputs, a function of (background, alphas or None, sh or None) that runs the raw backward)."""
    scene = configs.make_scene(1, count=count, width=side, height=side, device=device)
    scene["opacities"] = torch.full((count, 1), 0.05, device=device)
    scene["bg"] = torch.tensor([5.0, -3.0, 2.0], device=device)
    x = raster_inputs(scene)
    fwd = _rasterizer.rasterize_gaussians(
        x.background, x.means3d, x.colors, x.opacities, x.scales, x.rotations, x.scale_modifier, x.cov3d_precomp,
        x.viewmatrix, x.projmatrix, x.tan_fovx, x.tan_fovy, side, side, x.sh, x.degree, x.campos, False)
    num_rendered, _, _, alpha, radii, geom, binning, img = fwd[:8]
    assert num_rendered > 0
    g = torch.Generator().manual_seed(4)
    up = [torch.randn(c, side, side, generator=g).to(device) for c in (3, 1, 1)]

    def run(background, alphas=None, sh=None):
        return _rasterizer.rasterize_gaussians_backward(
            background, x.means3d, radii, x.colors, x.opacities, x.scales, x.rotations, x.scale_modifier,
            x.cov3d_precomp, x.viewmatrix, x.projmatrix, x.tan_fovx, x.tan_fovy, *up, None, None, None,
            x.sh if sh is None else sh, x.degree, x.campos, geom, num_rendered, binning, img,
            alpha if alphas is None else alphas)

    return x, alpha, run


def test_background_on_the_host_with_converted_images(device):
    x, alpha, run = _call(device)
    half = alpha.half()  # its float32 copy is as small as the background's
    want = run(x.background, half)
    got = run(x.background.cpu(), half)
    for a, b in zip(got, want):
        # the order of the float atomics: at most 64 pixels per sum
        assert bool(((a - b).abs() <= 1e-4 * b.abs().max() + 1e-12).all()) if b.numel() else a.shape == b.shape


@pytest.mark.parametrize("change", [1, -1, -47])
def test_sh_of_another_size_is_refused_before_the_launches(change, device, monkeypatch):
    x, _, run = _call(device)
    sh = torch.zeros(x.sh.numel() + change, device=device)
    called = []
    lib = _lib.load()
    real = lib.call
    monkeypatch.setattr(lib, "call", lambda name, *args: (called.append(name), real(name, *args))[1])
    with pytest.raises(RuntimeError):
        run(x.background, sh=sh)
    assert called == []
