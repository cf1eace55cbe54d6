"""The bucketed binning's running positions: scanned in place up to 4096 chunks of 256 Gaussians,
transposed beyond.  The lists must be those of the depth-then-tile sort bit for bit."""

from __future__ import annotations

import pytest
import torch

from gswarp_amd import _lib, _pipeline, configs
from helpers import gpu_forward, options

pytestmark = pytest.mark.gpu


def _pile(count, width, height, device):
    """`count` splats of a pixel or two, all of them in view."""
    scene = configs.make_scene(1, count=count, width=width, height=height, device=device)
    g = torch.Generator().manual_seed(count)
    pixel = 4.0 * 2.0 * scene["tanfovx"] / width
    means = torch.rand(count, 3, generator=g) * 2.0 - 1.0
    means[:, 0] *= 0.4 * width * pixel
    means[:, 1] *= 0.4 * height * pixel
    means[:, 2] *= 0.2
    scene["means3D"] = means.to(device)
    scene["scales"] = (pixel * (0.5 + torch.rand(count, 3, generator=g))).to(device)
    scene["opacities"] = torch.full((count, 1), 0.5, device=device)
    return scene


@pytest.mark.parametrize("count,width,height", [
    (1, 16, 16), (256, 130, 20), (257, 130, 140), (65_536, 400, 300), (65_537, 400, 300),
    (3000, 4080, 4080),                          # 32 x 32 super-tiles
    (1_048_576, 300, 260), (1_048_832, 300, 260),  # 4096 chunks, and more
])
def test_lists_match_the_depth_tile_sort(count, width, height, device, monkeypatch):
    scene = _pile(count, width, height, device)
    monkeypatch.setattr(_pipeline, "DEPTH_TILE_MIN_PAIRS_PER_GAUSSIAN", 0)
    monkeypatch.setattr(_pipeline, "BUCKET_SIZING", "always")
    outs = {}
    for flow in ("buckets", "depth_tile"):
        monkeypatch.setattr(_pipeline, "HEAVY_DATAFLOW", flow)
        print(f"[columns] N={count} {width}x{height} {flow}", flush=True)
        outs[flow] = gpu_forward(scene, options())["bins"]
    a, b = outs["buckets"], outs["depth_tile"]
    assert a.num_rendered == b.num_rendered >= count
    assert torch.equal(a.point_list, b.point_list)
    assert torch.equal(a.ranges, b.ranges)


@pytest.mark.parametrize("count", [5000, 1_572_864, 1_572_865])
def test_depth_order_in_wide_digits(count, device, monkeypatch):
    """Depths of 25 to 27 bits take a digit pass less in 9-bit digits, up to 1.5M Gaussians; equal depths keep
    their order."""
    width, height = 300, 260
    scene = _pile(count, width, height, device)
    g = torch.Generator().manual_seed(count + 1)
    depth = 2.0 + 7.0 * torch.rand(count, generator=g)
    depth[::7] = depth[0]
    depth = depth.to(device)
    scene["means3D"] *= (depth / 4.0)[:, None]  # the same place in the image
    scene["means3D"][:, 2] = depth - 4.0
    scene["scales"] *= (depth / 4.0)[:, None]
    monkeypatch.setattr(_pipeline, "DEPTH_TILE_MIN_PAIRS_PER_GAUSSIAN", 0)
    monkeypatch.setattr(_pipeline, "BUCKET_SIZING", "always")
    outs = {}
    for flow in ("buckets", "depth_tile"):
        monkeypatch.setattr(_pipeline, "HEAVY_DATAFLOW", flow)
        print(f"[wide digits] N={count} {flow}", flush=True)
        outs[flow] = gpu_forward(scene, options())
    pre = outs["buckets"]["pre"]
    bits = pre.depths[pre.radii > 0].view(torch.int32)
    assert (int(bits.max()) - int(bits.min()) + 1).bit_length() in (25, 26, 27)
    a, b = outs["buckets"]["bins"], outs["depth_tile"]["bins"]
    assert a.num_rendered == b.num_rendered >= count
    assert torch.equal(a.point_list, b.point_list) and torch.equal(a.ranges, b.ranges)
    # scratch for 8-bit digits of 4096-key tiles only: the narrow digits, a pass more
    lib = _lib.load()
    real = lib.gs_bin_buckets_workspace_bytes
    short = int(lib.gs_sort_scratch_bytes(count)) - ((count + 4095) // 4096 + 1) * 1024
    assert short > 0
    monkeypatch.setattr(_pipeline, "HEAVY_DATAFLOW", "buckets")
    monkeypatch.setattr(lib, "gs_bin_buckets_workspace_bytes", lambda *args: real(*args) - short)
    assert torch.equal(gpu_forward(scene, options())["bins"].point_list, b.point_list)


def test_workspace_of_the_least_size_serves(device, monkeypatch):
    """The depth sort's fast split wants more scratch than 4096-key tiles; without it the lists are the same."""
    from gswarp_amd import _lib

    count = 20_000
    scene = _pile(count, 130, 140, device)
    monkeypatch.setattr(_pipeline, "DEPTH_TILE_MIN_PAIRS_PER_GAUSSIAN", 0)
    monkeypatch.setattr(_pipeline, "BUCKET_SIZING", "always")
    expected = gpu_forward(scene, options())["bins"].point_list
    lib = _lib.load()
    real = lib.gs_bin_buckets_workspace_bytes
    least = ((count + 4095) // 4096 + 1) * 1024
    short = int(lib.gs_sort_scratch_bytes(count)) - least
    assert short > 0
    monkeypatch.setattr(lib, "gs_bin_buckets_workspace_bytes", lambda *a: real(*a) - short)
    assert torch.equal(gpu_forward(scene, options())["bins"].point_list, expected)
    monkeypatch.setattr(lib, "gs_bin_buckets_workspace_bytes", lambda *a: real(*a) - short - 256)
    with pytest.raises(RuntimeError):
        gpu_forward(scene, options())
