"""The render backward's segmented walk (gs_render_bwd_ws) against the oracle.

Images of few tiles have a slice's walk cut into segments of 128 entries or
more, at most 32 (T <= 1024 tiles); quadrants up to 12 pairs per Gaussian,
halves above.  Lists are made just below, at and above one, two and 32
segments; the bar is the per-element one of test_gpu_parity.py.
"""

from __future__ import annotations

import pytest
import torch

from gswarp_amd import _lib, configs
from test_gpu_parity import _check_backward


def _pile(count: int, side: int, sigma_px: float, device) -> dict:
    """`count` faint splats of about `sigma_px` pixels scattered over a side x side image: no pixel
    stops, so every walk reaches the last splats of its tile's list."""
    scene = configs.make_scene(1, count=count, width=side, height=side, device=device)
    g = torch.Generator().manual_seed(count)
    focal = side / (2.0 * scene["tanfovx"])
    half = 0.5 * side * 4.0 / focal
    means = torch.rand(count, 3, generator=g) * 2.0 - 1.0
    means[:, :2] *= half
    means[:, 2] *= 0.2
    scene["means3D"] = means.to(device)
    scale = sigma_px * 4.0 / focal
    scene["scales"] = (scale * (0.8 + 0.4 * torch.rand(count, 3, generator=g))).to(device)
    scene["opacities"] = (0.006 + 0.03 * torch.rand(count, 1, generator=g)).to(device)
    return scene


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 64, 127, 128, 129, 256, 257, 4095, 4097, 4300])
def test_quadrant_segments_match_oracle(count, device):
    assert _lib.load().gs_render_bwd_workspace_bytes(16, 16, count, count) > 0
    _check_backward(_pile(count, 16, 1.5, device))


@pytest.mark.gpu
@pytest.mark.parametrize("count,compute_depth", [(100, True), (129, False), (300, True)])
def test_half_segments_match_oracle(count, compute_depth, device):
    # splats over every tile of a ragged 5 x 5 tile image: 25 pairs each
    _check_backward(_pile(count, 67, 40.0, device), compute_depth=compute_depth)


def test_workspace_only_where_the_walk_is_cut():
    lib = _lib.load()
    needs = lambda w, h, n, r: lib.gs_render_bwd_workspace_bytes(w, h, n, r) > 0
    assert needs(640, 640, 1_000_000, 9_000_000) and needs(640, 640, 300_000, 9_000_000)  # 1600 tiles
    assert needs(800, 800, 300_000, 500_001) and not needs(800, 800, 900_000, 1_250_001)  # 2500 tiles
    assert needs(800, 800, 300_000, 1_250_001) and not needs(800, 800, 100_000, 1_250_001)
    assert not needs(1280, 720, 300_000, 300_000)  # 3600 tiles
    assert not needs(640, 640, 1000, 0) and not needs(0, 640, 1000, 1000)
    # 64 (a, b) pairs for each of a quadrant's segments but the first, and its length
    assert lib.gs_render_bwd_workspace_bytes(16, 16, 10, 10) == 4 * (31 * 64 * 8 + 4)
