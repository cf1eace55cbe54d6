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
from helpers import gpu_forward, options
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


def _sums(scene, out, alpha, n_contrib):
    """(segmented, whole) render gradients, (N, 10), of a forward; the segmented walk's workspace is filled
    with NaN."""
    pre, bins, device = out["pre"], out["bins"], alpha.device
    H, W, N, R = scene["height"], scene["width"], scene["means3D"].shape[0], bins.num_rendered
    g = torch.Generator().manual_seed(9)
    grads = [torch.randn(c, H, W, generator=g).to(device) for c in (3, 1, 1)]
    lib = _lib.load()
    size = lib.gs_render_bwd_workspace_bytes(W, H, N, R)
    assert size > 0
    sums = []
    for ws in (torch.full((size // 4,), float("nan"), device=device), None):
        acc = torch.zeros((N, 10), device=device)
        lib.call("gs_render_bwd_ws", W, H, N, R, bins.ranges.data_ptr(), bins.point_list.data_ptr(),
                 pre.records.data_ptr(), scene["bg"].data_ptr(), alpha.data_ptr(), n_contrib.data_ptr(),
                 *(t.data_ptr() for t in grads), 1, acc.data_ptr(), None, _lib.ptr(ws), size if ws is not None else 0,
                 torch.cuda.current_stream(device).cuda_stream)
        sums.append(acc)
    torch.cuda.synchronize()
    return sums


def _walks(scene, limit: int, device):
    """_sums of a scene whose blocks of 8 x 8 pixels are given walks of at most `limit` entries, but for one
    pixel each whose alpha is 1."""
    out = gpu_forward(scene, options())
    n_contrib = out["res"].n_contrib.view(scene["height"], scene["width"]).clamp(max=limit)
    alpha = out["res"].alpha.clone()
    at = (slice(3, None, 8), slice(5, None, 8))
    n_contrib[at] = out["res"].n_contrib.view_as(n_contrib)[at]
    alpha[0][at] = 1.0
    return _sums(scene, out, alpha, n_contrib)


def _assert_close(segmented, whole):
    # a pixel's state is a product and a sum over a few hundred entries, each rounded to 2^-24 of it, and a
    # Gaussian's sum has at most a few hundred terms of either sign
    tol = 1e-4 * whole.abs().amax(dim=0, keepdim=True) + 1e-12
    assert bool(((segmented - whole).abs() <= tol).all())


@pytest.mark.gpu
@pytest.mark.parametrize("count,side,sigma,pixels", [(400, 16, 6.0, "quadrants"), (400, 67, 40.0, "halves")])
@pytest.mark.parametrize("limit", [0, 1, 90, 128, 129, 300])
def test_opaque_pixel_with_the_longest_walk(count, side, sigma, pixels, limit, device):
    """A pixel of alpha 1 blends nothing: where it alone has entries in the last segments, those segments
    pass the other pixels' state on unchanged."""
    _assert_close(*_walks(_pile(count, side, sigma, device), limit, device))


@pytest.mark.gpu
@pytest.mark.parametrize("count,side,sigma,pixels", [(700, 16, 2.0, "quadrants"), (1200, 67, 25.0, "halves")])
def test_pixels_of_a_block_end_in_different_segments(count, side, sigma, pixels, device):
    """Opaque splats in front cover a column of each of the first tile's blocks: their pixels end after some tens of
    entries, beside pixels whose walks reach the list's end."""
    scene = _pile(count, side, sigma, device)
    g = torch.Generator().manual_seed(count)
    pixel = 8.0 * scene["tanfovx"] / side
    front = torch.rand(120, 3, generator=g).to(device)
    z = -0.3 - 0.1 * front[:, 2]
    # the view mirrors x and y
    scene["means3D"][:120, 0] = (0.5 * side - 4.0 - 8.0 * front[:, 0].round()) * pixel * (4.0 + z) / 4.0
    scene["means3D"][:120, 1] = (0.5 * side - 16.0 * front[:, 1]) * pixel * (4.0 + z) / 4.0
    scene["means3D"][:120, 2] = z
    scene["scales"][:120] = pixel
    scene["opacities"][:120] = 0.99
    out = gpu_forward(scene, options())
    ends = out["res"].n_contrib.view(side, side)[:16, :8]
    print(f"[ends] {pixels} {int(ends.min())} {int(ends.max())} of "
          f"{int(out['bins'].ranges[0, 1] - out['bins'].ranges[0, 0])}", flush=True)
    assert int(ends.min()) <= 128 and int(ends.max()) > 4 * 128
    _assert_close(*_sums(scene, out, out["res"].alpha, out["res"].n_contrib))
    _check_backward(scene)


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


def test_no_more_segments_than_the_lists_fill():
    """Segments of 128 entries for lists of 32 times the mean length, but where there are fewer than 128 tiles."""
    lib = _lib.load()
    size = lib.gs_render_bwd_workspace_bytes
    cut = lambda tiles, segments: tiles * ((segments - 1) * 256 * 8 + 4 * 4)
    assert size(512, 512, 3000, 4096) == 0  # 1024 tiles, mean 4
    assert size(512, 512, 3000, 4097) == cut(1024, 2)
    assert size(512, 512, 30_000, 4096 * 31) == cut(1024, 31)
    assert size(512, 512, 1_000_000, 4096 * 100) == cut(1024, 32)
    assert size(800, 800, 100, 200) == 0 and size(800, 800, 100_000, 10_001) == cut(2500, 2)
    assert size(176, 176, 100, 200) == 0  # 121 tiles
    assert size(128, 128, 100, 200) == cut(64, 2) and size(32, 32, 100, 200) == cut(4, 32)


def test_short_workspace_is_refused():
    """As short scratch is by the sorts and the binning, before anything is launched."""
    lib = _lib.load()
    size = lib.gs_render_bwd_workspace_bytes(64, 64, 1000, 5000)
    at = 4096  # never read: the call returns before its launches
    call = lambda ws, nbytes: lib.gs_render_bwd_ws(64, 64, 1000, 5000, at, at, at, at, at, at, at, at, at, 1, at, None,
                                                   ws, nbytes, None)
    assert size > 0 and call(at, size - 1) == -3 and call(at, 0) == -3
    assert "scratch" in lib.status_string(-3)
    assert call(at + 4, size) not in (0, -3)  # misaligned


@pytest.mark.gpu
@pytest.mark.parametrize("count", [500, 1500])
def test_segments_longer_than_128_entries_match_oracle(count, device):
    """A small object: its lists are longer than the cut is made for."""
    scene = _pile(count, 256, 3.0, device)
    scene["means3D"][:, :2] *= 0.05
    out = gpu_forward(scene, options())["bins"]
    longest = int((out.ranges[:, 1] - out.ranges[:, 0]).max())
    segments = _lib.load().gs_render_bwd_workspace_bytes(256, 256, count, out.num_rendered) // (256 * 2048) + 1
    assert 1 < segments and longest > 128 * segments
    _check_backward(scene)
