"""The state classes whose arrays lie in one allocation are the plain state dataclasses to their holders:
instances of them, with fields that can be set, replaced, copied and pickled."""

from __future__ import annotations

import copy
import dataclasses
import pickle

import pytest
import torch

from gswarp_amd import _state

P, T, PIXELS = 5, 3, 7
SPANS = [("records", torch.float32, (P, 12), 48 * P), ("coverage", torch.int32, (P, 4), 16 * P),
         ("depths", torch.float32, (P,), 4 * P), ("tiles_touched", torch.int32, (P,), 4 * P),
         ("clamped", torch.uint8, (P,), P), ("ranges", torch.int32, (T, 2), 8 * T),
         ("tile_order", torch.int32, (T,), 4 * T), ("n_contrib", torch.int32, (PIXELS,), 4 * PIXELS)]


def _state_of(rendered: bool = True):
    arena = _state.StateArena(SPANS, torch.device("cpu"))
    arena.buffer.copy_(torch.arange(arena.buffer.numel()) % 251)
    pre = _state.ArenaPreprocessOutputs.within(arena, torch.ones(P, dtype=torch.int32), torch.zeros(P, 2),
                                               torch.zeros(P, 3), torch.zeros(P, 3), 1)
    bins = _state.ArenaBinningState.within(arena, 3, 1, torch.zeros(4, dtype=torch.int32), 4, _state.KeyLayout(1, 2, 3),
                                           rendered)
    return _state.ArenaForwardState.within(arena, pre, bins, None)


PLAIN = {"preprocess": _state.PreprocessOutputs, "binning": _state.BinningState}


def _parts(state):
    return {"": state, "preprocess": state.preprocess, "binning": state.binning}


def _tensors(part):
    return {f.name: getattr(part, f.name) for f in dataclasses.fields(part)
            if isinstance(getattr(part, f.name), torch.Tensor)}


def test_instances_of_the_plain_classes():
    for name, part in _parts(_state_of()).items():
        assert isinstance(part, PLAIN.get(name, _state.ForwardState))


def test_every_array_has_its_address():
    for part in _parts(_state_of()).values():
        for name, tensor in _tensors(part).items():
            assert part.address(name) == tensor.data_ptr(), name
            assert getattr(part, name) is tensor
    state = _state_of()
    assert state.preprocess.band_store is None and state.preprocess.address("band_store") is None


def test_no_address_is_kept():
    """An address is that of the memory the state holds now, not of the memory it had when it was made."""
    state = _state_of()
    assert not any(isinstance(getattr(state.binning.arena, s), int) for s in _state.StateArena.__slots__)


def test_fields_can_be_set():
    for name, part in _parts(_state_of()).items():
        for field in dataclasses.fields(part):
            old = getattr(part, field.name)
            new = old.clone() if isinstance(old, torch.Tensor) else old
            setattr(part, field.name, new)
            assert getattr(part, field.name) is new
            if isinstance(new, torch.Tensor):
                assert part.address(field.name) == new.data_ptr()
    pre = _state_of().preprocess
    pre.depths = None
    assert pre.address("depths") is None


@pytest.mark.parametrize("rendered", [True, False])
def test_tile_order_only_once_written(rendered):
    bins = _state_of(rendered).binning
    assert (bins.tile_order is not None) == (bins.address("tile_order") is not None) == rendered
    bins.ensure_tile_order(T)
    assert bins.tile_order.shape == (T,) and bins.address("tile_order") == bins.tile_order.data_ptr()


@pytest.mark.parametrize("how", ["copy", "deepcopy", "pickle", "replace", "torch"])
def test_copies(how, tmp_path):
    for part in _parts(_state_of()).values():
        if how == "copy":
            other = copy.copy(part)
        elif how == "deepcopy":
            other = copy.deepcopy(part)
        elif how == "pickle":
            other = pickle.loads(pickle.dumps(part))
        elif how == "torch":
            torch.save(part, tmp_path / "state.pt")
            other = torch.load(tmp_path / "state.pt", weights_only=False)
        else:
            other = dataclasses.replace(part)
        shared = how in ("copy", "replace")
        for name, tensor in _tensors(part).items():
            got = getattr(other, name)
            assert got.dtype == tensor.dtype and torch.equal(got.view(torch.uint8), tensor.view(torch.uint8)), name
            assert (got.data_ptr() == tensor.data_ptr()) == shared, name
            assert other.address(name) == got.data_ptr()
        if not shared:  # a copied array does not keep the other arrays' memory
            assert sum(t.untyped_storage().nbytes() for t in _tensors(other).values()) <= \
                sum(t.numel() * t.element_size() for t in _tensors(part).values())
