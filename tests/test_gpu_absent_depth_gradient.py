"""The render backward without an upstream depth gradient (null: the depth terms
left out of the walk) against one of zeros, in every shape of the walk."""

from __future__ import annotations

import pytest
import torch

from gswarp_amd import _lib, configs
from helpers import gpu_forward, options

# quadrants in segments, halves in segments, halves, whole tiles
SHAPES = {"quadrants": (2, 20_000, 203, 117), "halves_segments": (3, 3_000, 203, 117),
          "halves": (2, 60_000, 1000, 800), "whole": (3, 60_000, 1000, 800)}


@pytest.mark.gpu
@pytest.mark.parametrize("segments", [True, False])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_absent_depth_gradient_is_zero(shape, segments, device):
    config, count, width, height = SHAPES[shape]
    scene = configs.make_scene(config, count=count, width=width, height=height, device=device)
    out = gpu_forward(scene, options())
    lib, bins, res = _lib.load(), out["bins"], out["res"]
    g = torch.Generator().manual_seed(4)
    color = torch.randn(3, height, width, generator=g).to(device)
    zero = torch.zeros(1, height, width, device=device)
    nbytes = lib.gs_render_bwd_workspace_bytes(width, height, count, bins.num_rendered) if segments else 0
    sums = []
    for depth in (zero, None):
        ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device=device)
        gg = torch.zeros(count, 10, device=device)
        assert lib.gs_render_bwd_ws(
            width, height, count, bins.num_rendered, bins.ranges.data_ptr(), bins.point_list.data_ptr(),
            out["pre"].records.data_ptr(), scene["bg"].data_ptr(), res.alpha.data_ptr(), res.n_contrib.data_ptr(),
            color.data_ptr(), None if depth is None else depth.data_ptr(), None, 1, gg.data_ptr(), None,
            ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream(device).cuda_stream) == 0
        torch.cuda.synchronize()
        sums.append(gg)
    assert float(sums[0].abs().max()) > 0 and not bool(sums[1][:, 9].any())
    # the same terms; the atomics' order differs between runs (a few hundred float32 additions)
    scale = sums[0].abs().amax(0)
    assert bool(((sums[0] - sums[1]).abs() <= 1e-4 * scale + 1e-30).all())
