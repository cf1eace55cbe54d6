"""The forward render in 4x4-pixel blocks against the oracle, bit for bit: list
lengths around its steps of four records and batches of 64, ragged images, and
opaque piles whose pixels stop at every position of a step."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from gswarp_amd import configs
from helpers import gpu_forward, options, oracle_forward, to_np
from test_gpu_parity import _check_forward

pytestmark = pytest.mark.gpu


def _pile(count, width, height, opacity, device):
    """`count` splats of a few pixels over the image, opacities in `opacity`."""
    scene = configs.make_scene(1, count=count, width=width, height=height, device=device)
    g = torch.Generator().manual_seed(100 * count + width)
    pixel = 4.0 * 2.0 * scene["tanfovx"] / width
    means = torch.rand(count, 3, generator=g) * 2.0 - 1.0
    means[:, 0] *= 0.5 * width * pixel
    means[:, 1] *= 0.5 * height * pixel
    means[:, 2] *= 0.2
    scene["means3D"] = means.to(device)
    scene["scales"] = (pixel * (1.0 + 4.0 * torch.rand(count, 3, generator=g))).to(device)
    lo, hi = opacity
    scene["opacities"] = (lo + (hi - lo) * torch.rand(count, 1, generator=g)).to(device)
    scene["bg"] = torch.tensor((0.2, 0.5, 0.9), device=device)
    return scene


@pytest.mark.parametrize("opacity", [(0.01, 0.2), (0.5, 1.0)])
@pytest.mark.parametrize("count", [1, 3, 4, 5, 63, 64, 65, 128, 131, 400])
def test_blocks_match_oracle(count, opacity, device):
    _check_forward(_pile(count, 21, 13, opacity, device), options())


@pytest.mark.parametrize("width,height", [(1, 1), (4, 4), (5, 3), (16, 16), (17, 33)])
def test_block_edges_match_oracle(width, height, device):
    scene = _pile(200, width, height, (0.05, 0.9), device)
    _check_forward(scene, options())
    _check_forward(scene, options(compute_depth=False))


@pytest.mark.parametrize("count", [150, 700])
def test_light_images_match_oracle(count, device):
    """Both sides of the least number of pairs that blocks take on more than 512 tiles."""
    scene = _pile(count, 400, 336, (0.05, 0.9), device)
    _check_forward(scene, options())
    pairs = gpu_forward(scene, options())["bins"].num_rendered
    assert (pairs < 4 * 25 * 21) == (count == 150)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_non_finite_colour_stays_with_its_pixels(value, device):
    """A step evaluates four records at a pixel; one that the pixel does not blend adds nothing, whatever its colour."""
    scene = _pile(131, 37, 29, (0.05, 0.5), device)
    scene["colors_precomp"] = torch.rand(131, 3, generator=torch.Generator().manual_seed(5)).to(device)
    scene["colors_precomp"][::40] = value
    got = to_np(gpu_forward(scene, options(), colors=True)["res"].color)
    expected = oracle_forward(scene, compute_depth=True, colors=True)[1]["fwd"]["color"]
    finite = np.isfinite(expected)
    assert 0 < finite.sum() < finite.size
    assert np.array_equal(np.isfinite(got), finite)
    assert np.array_equal(got[finite], expected[finite])
