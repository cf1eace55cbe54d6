"""The typed forward's ordinary course (_pipeline._forward_arena) against the
general one over the forms of input it takes: the same outputs bit for bit
and the same gradients up to the order of the float atomics."""

from __future__ import annotations

import copy

import pytest
import torch

from helpers import options, raster_inputs
from gswarp_amd import _pipeline, _validation, _workspace, configs, rasterizer, rasterizer_flow
from gswarp_amd.methods import mip_3dgs

pytestmark = pytest.mark.gpu


def _strided(t):
    """The same values, not contiguous."""
    return torch.stack([t, torch.zeros_like(t)], dim=-1)[..., 0]


def _misaligned(t):
    """The same values, contiguous, 4 bytes past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t.reshape(-1)
    return buf[1:].view(t.shape)


def _call(form: str, config: int, device):
    scene = configs.make_scene(config, seed=2, count=9_000, width=203, height=117, device=device)
    fields = dict(image_height=117, image_width=203, tanfovx=scene["tanfovx"], tanfovy=scene["tanfovy"],
                  bg=scene["bg"] + 0.25, scale_modifier=1.0, viewmatrix=scene["viewmatrix"],
                  projmatrix=scene["projmatrix"], sh_degree=3, campos=scene["campos"], prefiltered=False)
    leaves = {k: scene[k] for k in ("means3D", "scales", "rotations", "opacities", "shs")}
    leaves["means2D"] = torch.zeros_like(scene["means3D"])
    module, make = rasterizer, rasterizer.GaussianRasterizationSettings
    if form == "colors":
        leaves["colors_precomp"] = leaves.pop("shs")[:, 0].abs().contiguous()
    elif form == "cov":
        n = leaves["means3D"].shape[0]
        s2 = leaves.pop("scales") ** 2
        leaves.pop("rotations")
        cov = torch.zeros(n, 6, device=device)
        cov[:, [0, 3, 5]] = s2
        leaves["cov3D_precomp"] = cov
    elif form == "few_coefficients":
        leaves["shs"] = leaves["shs"][:, :4].contiguous()
        fields["sh_degree"] = 1
    elif form == "strided":
        leaves = {k: _strided(v) for k, v in leaves.items()}
        fields["viewmatrix"] = fields["viewmatrix"].t().contiguous().t()
    elif form == "misaligned":
        leaves = {k: _misaligned(v) for k, v in leaves.items()}
    elif form == "flow":
        module, make = rasterizer_flow, rasterizer_flow.GaussianRasterizationSettings
    elif form == "mip":
        module, make = None, mip_3dgs.MipGaussianRasterizationSettings
        fields["filter_variance"] = 0.3
    elif form == "warp_radix":
        fields["binning_sort_mode"] = "warp_radix"
    raster = (mip_3dgs.MipGaussianRasterizer if form == "mip" else module.GaussianRasterizer)(make(**fields))
    leaves = {k: v.detach().requires_grad_(True) for k, v in leaves.items()}

    def run():
        out = raster(**leaves)
        flat = list(out) if form == "flow" else [out[0], out[1], *out[2]]
        grads = torch.autograd.grad([flat[0].sum() + (flat[2] if form == "flow" else out[2].depth).sum()],
                                    list(leaves.values()))
        return [t.detach() for t in flat], grads

    return run


@pytest.mark.parametrize("form", ["sh", "colors", "cov", "few_coefficients", "strided", "misaligned", "flow", "mip",
                                  "warp_radix"])
@pytest.mark.parametrize("config,hint", [(2, 9_000), (2, 1), (3, 1_000_000)])
def test_arena_forward_equals_general(form, config, hint, device, monkeypatch):
    """hint: the last forward's pair count, for a provision that fits, one
    that is declined, and the bucketed binning."""
    run = _call(form, config, device)
    taken = []
    real = _pipeline._forward_arena

    def spy(*args, **kw):
        result = real(*args, **kw)
        taken.append(result is not None)
        return result

    monkeypatch.setattr(_pipeline, "_forward_arena", spy)
    _workspace.note_pairs(device, hint)
    out, grads = run()
    assert taken == [True]
    monkeypatch.setattr(_pipeline, "_forward_arena", lambda *a, **k: None)
    _workspace.note_pairs(device, hint)
    want, want_grads = run()
    for a, b in zip(out, want):
        assert torch.equal(a, b)
    for a, b in zip(grads, want_grads):
        assert a.shape == b.shape
        # the atomics' order: a few hundred float32 additions per element
        assert float((a - b).abs().max()) <= 1e-4 * float(b.abs().max()) + 1e-12


def test_backward_from_a_copied_state(device):
    """The copy is on its own: the state it was made from is gone, and its memory overwritten, by the backward."""
    scene = configs.make_scene(2, seed=3, count=5_000, width=120, height=90, device=device)
    inputs, opts = raster_inputs(scene), options()
    _workspace.note_pairs(device, 5_000)
    upstream = torch.randn(3, 90, 120, generator=torch.Generator().manual_seed(1)).to(device)

    def grads(copied: bool):
        result = _pipeline.forward(inputs, opts)
        state = result.state
        if copied:
            state = copy.deepcopy(state)
            result.state.binning.arena.buffer.fill_(255)
        return _pipeline.backward(inputs, result.radii, result.alpha, upstream, None, None, None, None, None, opts,
                                  state)

    for a, b in zip(grads(True), grads(False)):
        assert a.shape == b.shape
        if b.numel():  # the atomics' order
            assert float((a - b).abs().max()) <= 1e-4 * float(b.abs().max()) + 1e-12


def test_first_forward_takes_the_general_course(device):
    _workspace.clear_caches()
    run = _call("sh", 2, device)
    first, _ = run()
    again, _ = run()
    for a, b in zip(first, again):
        assert torch.equal(a, b)


def test_one_pass_validation_refuses_what_the_staged_checks_refuse(device):
    scene = configs.make_scene(1, count=50, width=64, height=64, device=device)
    settings = rasterizer.GaussianRasterizationSettings(64, 64, 0.5, 0.5, scene["bg"], 1.0, scene["viewmatrix"],
                                                        scene["projmatrix"], 3, scene["campos"], False)
    empty = torch.empty(0, device=device)
    args = dict(means3D=scene["means3D"], means2D=torch.zeros_like(scene["means3D"]), sh=scene["shs"],
                colors_precomp=empty, opacities=scene["opacities"], scales=scene["scales"],
                rotations=scene["rotations"], cov3Ds_precomp=empty)

    def plain(settings=settings, **change):
        values = {**args, **change}
        return _validation._plainly_valid(*values.values(), settings)

    def staged(settings=settings, **change):
        values = {**args, **change}
        try:
            _validation.validate_rasterizer_inputs(*values.values(), settings)
        except ValueError:
            return False
        return True

    assert plain() and staged()
    bad = torch.zeros
    changes = [dict(means3D=None), dict(means3D=args["means3D"].cpu()), dict(means3D=args["means3D"].double()),
               dict(means3D=bad(50, 4, device=device)), dict(means2D=bad(49, 3, device=device)),
               dict(means2D=args["means2D"].half()), dict(opacities=bad(49, 1, device=device)),
               dict(opacities=args["opacities"].cpu()), dict(sh=empty), dict(sh=args["sh"][:, :4].contiguous()),
               dict(sh=bad(50 * 48 + 1, device=device)), dict(colors_precomp=bad(50, 3, device=device)),
               dict(scales=empty), dict(rotations=empty), dict(rotations=bad(50, 3, device=device)),
               dict(cov3Ds_precomp=bad(50, 6, device=device)), dict(scales=args["scales"].double()),
               dict(sh=empty, colors_precomp=bad(50, 4, device=device)), dict(colors_precomp=None)]
    for change in changes:
        assert not plain(**change) and not staged(**change), change
    nan = float("nan")
    for field in (dict(image_height=0), dict(image_width=64.0), dict(image_height=1 << 20, image_width=1 << 20),
                  dict(tanfovx=nan), dict(tanfovy=0.0), dict(scale_modifier=float("inf")), dict(sh_degree=-1),
                  dict(sh_degree=1.0), dict(bg=bad(4, device=device)), dict(campos=scene["campos"].cpu()),
                  dict(viewmatrix=bad(16, device=device)), dict(projmatrix=None)):
        changed = settings._replace(**field)
        assert not plain(changed) and not staged(changed), field
    # refused by the one pass only because it leaves them to the staged checks
    assert not plain(settings._replace(debug=True)) and staged(settings._replace(debug=True))
