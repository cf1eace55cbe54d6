"""Typed state carried from the forward stages to the backward.

Counterparts of gswarp/_internal/backends/warp/state.py:48-110.  The render
stage reads one packed 48-byte record per Gaussian (``records``) instead of
separate points_xy / conic_opacity / features / depths arrays.
"""

from __future__ import annotations

from dataclasses import dataclass, field, fields

import torch


@dataclass(slots=True)
class PreprocessOutputs:
    radii: torch.Tensor  # (N,) int32
    depths: torch.Tensor  # (N,) view-space z of visible Gaussians, 0 otherwise
    proj_2d: torch.Tensor  # (N, 2) pixel-space centre (= the reference's points_xy_image)
    conic_2d: torch.Tensor  # (N, 3)
    conic_2d_inv: torch.Tensor  # (N, 3) 2D covariance incl. the 0.3 dilation
    tiles_touched: torch.Tensor  # (N,) int32
    records: torch.Tensor  # (N, 12) fp32 render records
    clamped: torch.Tensor  # (N,) uint8 SH clamp bits
    coverage_mode: int = 1
    geom: torch.Tensor | None = None  # raw-ABI byte buffer that records and clamped are views of
    coverage: torch.Tensor | None = None  # (N, 4) int32 cover words for the emission, or None (re-derived)
    band_store: torch.Tensor | None = None  # int32 coverage bands of the banded Gaussians, or None
    # gs_scan_tiles_onepass state that the preprocess prepared (serves one scan), or None
    scan_state: torch.Tensor | None = None

    def address(self, name: str) -> int | None:
        tensor = getattr(self, name)
        return None if tensor is None else tensor.data_ptr()


@dataclass(slots=True)
class KeyLayout:
    """Fields of the 64-bit binning key, from high to low:
    tile | float_bits(depth) - depth_min (depth_bits wide) | point index (value_bits wide, 0 = not packed)."""

    depth_min: int = 0
    depth_bits: int = 32
    value_bits: int = 0

    @property
    def tile_shift(self) -> int:
        return self.depth_bits + self.value_bits


@dataclass(slots=True)
class RenderImages:
    """Forward render outputs allocated before the binning, so that the binning
    call can launch the render into them."""

    background: torch.Tensor  # (3,) fp32, contiguous
    color: torch.Tensor  # (3, H, W)
    depth: torch.Tensor  # (1, H, W)
    alpha: torch.Tensor  # (1, H, W)
    n_contrib: torch.Tensor  # (H*W,) int32
    compute_depth: bool = True


@dataclass(slots=True)
class BinningState:
    grid_x: int
    grid_y: int
    point_list: torch.Tensor  # (R,) int32
    ranges: torch.Tensor  # (T, 2) int32
    num_rendered: int
    sorted_keys: torch.Tensor | None = None  # (R,) int64 sorted binning keys (see KeyLayout)
    key_layout: KeyLayout = field(default_factory=KeyLayout)
    buffer: torch.Tensor | None = None  # raw-ABI (R + 2T) int32 buffer that point_list and ranges are views of
    rendered: bool = False  # the standard forward render was launched with the binning (RenderImages)
    tile_order: torch.Tensor | None = None  # (T,) int32 buffer the forward render was given (gs_tile_order)

    def address(self, name: str) -> int | None:
        tensor = getattr(self, name)
        return None if tensor is None else tensor.data_ptr()

    def ensure_tile_order(self, num_tiles: int) -> None:
        if self.tile_order is None:
            self.tile_order = torch.empty((max(num_tiles, 1),), dtype=torch.int32, device=self.ranges.device)

    def decode_keys(self) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        """(tile id, depth float bits, sort field = tile and depth fields as one
        non-negative int64) of every sorted pair, from sorted_keys."""
        k = self.sorted_keys
        lay = self.key_layout
        field_ = (k >> lay.value_bits) & ((1 << (64 - lay.value_bits)) - 1) if lay.value_bits else k
        tile = (k >> lay.tile_shift) & ((1 << (64 - lay.tile_shift)) - 1)
        depth = (field_ & ((1 << lay.depth_bits) - 1)) + lay.depth_min
        return tile, depth, field_


@dataclass(slots=True)
class RenderStageResult:
    color: torch.Tensor
    depth: torch.Tensor
    alpha: torch.Tensor
    n_contrib: torch.Tensor
    aux: tuple[torch.Tensor, ...] = ()


@dataclass(slots=True)
class ForwardState:
    preprocess: PreprocessOutputs
    binning: BinningState
    n_contrib: torch.Tensor
    # (N, 10) float32 gradient accumulator that the forward render zeroed on
    # its way (None when the forward made none); one backward takes it
    grad_gauss: torch.Tensor | None = None

    def address(self, name: str) -> int:
        return getattr(self, name).data_ptr()


class StateArena:
    """One device allocation for the arrays that a typed forward keeps for its
    backward.  The stages and the backward need their addresses only; a
    tensor view is made when one is asked for, which spares an allocation or a
    view of each on every call.  A view that is kept keeps the whole
    allocation (a clone does not)."""

    __slots__ = ("buffer", "spans")

    def __init__(self, spans, device: torch.device):
        """spans: (name, dtype, shape, bytes) of each array; every array starts on a 256-byte boundary."""
        self.spans = {}
        at = 0
        for name, dtype, shape, nbytes in spans:
            self.spans[name] = (at, dtype, shape, nbytes)
            at += (nbytes + 255) & ~255
        self.buffer = torch.empty((at,), dtype=torch.uint8, device=device)

    def offset(self, name: str) -> int:
        return self.spans[name][0]

    def view(self, name: str) -> torch.Tensor:
        at, dtype, shape, nbytes = self.spans[name]
        return self.buffer[at:at + nbytes].view(dtype).view(shape)


def _arena_field(name: str) -> property:
    """A dataclass field whose array lies in the arena until another is set."""

    def get(self):
        if name not in self.own:
            self.own[name] = self.arena.view(name) if name in self.arena.spans else None
        return self.own[name]

    def put(self, value):
        try:
            self.own[name] = value
        except AttributeError:  # the dataclass's constructor, which gives every array
            self.arena, self.own = None, {name: value}

    return property(get, put)


class _InArena:
    """What makes a state dataclass one whose _arena_field arrays lie in
    ``arena``; ``own`` holds the views made of them and what was set in their
    place.  To its holder it is the dataclass ``plain``: it is made by
    ``within``, or by the dataclass's own constructor (dataclasses.replace)
    with every array given; copies and pickles are plain ones."""

    __slots__ = ()
    plain: type

    def address(self, name: str) -> int | None:
        if name not in self.own and self.arena is not None:
            span = self.arena.spans.get(name)
            if span is not None:
                return self.arena.buffer.data_ptr() + span[0]
        return super().address(name)

    def _values(self) -> dict:
        return {f.name: getattr(self, f.name) for f in fields(self)}

    def __copy__(self):
        return self.plain(**self._values())

    def __reduce__(self):
        # arrays of different types in one storage cannot be saved together
        values = [v.clone() if k in self.own and v is not None else v for k, v in self._values().items()]
        return self.plain, tuple(values)


class ArenaPreprocessOutputs(_InArena, PreprocessOutputs):
    """PreprocessOutputs whose arrays, but for the four that the forward returns, lie in an arena."""

    __slots__ = ("arena", "own")
    plain = PreprocessOutputs
    depths = _arena_field("depths")
    tiles_touched = _arena_field("tiles_touched")
    records = _arena_field("records")
    clamped = _arena_field("clamped")
    coverage = _arena_field("coverage")
    band_store = _arena_field("band_store")

    @classmethod
    def within(cls, arena: StateArena, radii, proj_2d, conic_2d, conic_2d_inv, coverage_mode: int):
        self = object.__new__(cls)
        self.arena, self.own = arena, {}
        self.radii, self.proj_2d, self.conic_2d, self.conic_2d_inv = radii, proj_2d, conic_2d, conic_2d_inv
        self.coverage_mode = coverage_mode
        self.geom = None
        self.scan_state = None  # the arena's has served its scan
        return self


class ArenaBinningState(_InArena, BinningState):
    """BinningState of the packed binning launched with the read-back, its ranges and tile order in an arena."""

    __slots__ = ("arena", "own")
    plain = BinningState
    ranges = _arena_field("ranges")
    tile_order = _arena_field("tile_order")

    @classmethod
    def within(cls, arena: StateArena, grid_x: int, grid_y: int, point_list, num_rendered: int, key_layout: KeyLayout,
               rendered: bool):
        self = object.__new__(cls)
        self.arena, self.own = arena, {}
        self.grid_x, self.grid_y = grid_x, grid_y
        self.point_list, self.num_rendered, self.key_layout = point_list, num_rendered, key_layout
        self.sorted_keys = self.buffer = None
        self.rendered = rendered
        if not rendered:
            self.tile_order = None  # until a render writes it
        return self

    def ensure_tile_order(self, num_tiles: int) -> None:
        if self.arena is None:
            super().ensure_tile_order(num_tiles)
        elif self.own.get("tile_order", self) is None:
            del self.own["tile_order"]  # the arena's


class ArenaForwardState(_InArena, ForwardState):
    """ForwardState with n_contrib in an arena."""

    __slots__ = ("arena", "own")
    plain = ForwardState
    n_contrib = _arena_field("n_contrib")

    @classmethod
    def within(cls, arena: StateArena, preprocess: PreprocessOutputs, binning: BinningState, grad_gauss):
        self = object.__new__(cls)
        self.arena, self.own = arena, {}
        self.preprocess, self.binning, self.grad_gauss = preprocess, binning, grad_gauss
        return self


@dataclass(slots=True)
class ForwardResult:
    num_rendered: int
    color: torch.Tensor
    depth: torch.Tensor
    alpha: torch.Tensor
    radii: torch.Tensor
    proj_2d: torch.Tensor
    conic_2d: torch.Tensor
    conic_2d_inv: torch.Tensor
    state: ForwardState | None
    aux: tuple[torch.Tensor, ...] = field(default_factory=tuple)
