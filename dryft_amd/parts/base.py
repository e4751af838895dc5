"""What a part is, and what it is told about a step.

A part (mixer, feed-forward, norm, position encoding, embedding, head) is built
from sizes and constants alone, names the tensors it needs by logical name, and
computes on packed rows. It never learns which model it is in: the model plan
maps logical tensor names to checkpoint names and wires the parts together.
"""

from __future__ import annotations

import functools
import inspect
from dataclasses import dataclass, field
from typing import Any

import torch

from ..weights.spec import MATRIX


@dataclass
class HostBatch:
    """The step as the host knows it (absent while a captured graph is replayed)."""

    slots: list[int]      # cache slot of each sequence, -1 for a sequence that sits out
    q_lens: list[int]     # rows each sequence occupies in this step
    starts: list[int]     # tokens each sequence had cached before the step


@dataclass
class StepContext:
    """Per-step facts shared by all parts. Index tensors are int32 on the device.

    Rows are the step's tokens, packed sequence after sequence. Row ``r`` belongs to
    sequence ``row_seq[r]`` in cache slot ``row_slot[r]`` (-1: takes no part) at
    position ``row_pos[r]``. ``cu_rows`` are prefix sums over sequences of rows;
    ``kv_len`` is each sequence's cached length after this step, ``seq_start`` before it.
    A part whose kernel walks the step in tiles of some number of rows asks ``tiles()``
    for the prefix sums of those.

    ``host`` is the step as the host knows it, or None while a captured step is replayed.
    A part must not let what it computes depend on whether ``host`` is there; it may only
    use it to do less (skip clearing rows that no sequence sitting out owns).
    """

    n_rows: int
    n_seqs: int
    dtype: torch.dtype
    device: torch.device
    row_seq: torch.Tensor
    row_slot: torch.Tensor
    row_pos: torch.Tensor
    cu_rows: torch.Tensor
    seq_slot: torch.Tensor
    q_len: torch.Tensor
    kv_len: torch.Tensor
    seq_start: torch.Tensor
    max_q_len: int                      # host bound on rows per sequence; 1 means a decoding step
    max_kv_len: int                     # host bound on any sequence's cached length after the step
    host: HostBatch | None = None
    positions: dict[str, Any] = field(default_factory=dict)   # name -> position encoding, tables ready
    embedded: torch.Tensor | None = None    # the embedding's output of this step's rows, for parts that come back to it
    tokens: torch.Tensor | None = None      # the step's token ids (int32, a row each), for parts that look them up
    # what a part of an earlier layer leaves for parts of later layers of the same step, by a name the plan gives
    # both (the values a first attention layer computed, which later ones lean on); emptied when a step begins
    shared: dict[str, Any] = field(default_factory=dict)
    _tiles: dict[int, tuple[torch.Tensor, int]] = field(default_factory=dict, repr=False)
    _kept: dict[Any, torch.Tensor] = field(default_factory=dict, repr=False)
    _counters: dict[int, torch.Tensor] = field(default_factory=dict, repr=False)

    def tiles(self, rows_per_tile: int) -> tuple[torch.Tensor, int]:
        """For kernels that walk the step tile by tile: ``(tile_cu, bound)``. ``tile_cu`` (int32, device,
        ``n_seqs + 1`` entries) holds the prefix sums over the sequences of the tiles of ``rows_per_tile`` rows that
        their rows of this step fill (a sequence that sits out fills none); ``bound`` is what the host knows the
        total not to exceed (a grid size). Computed when first asked for, once per tile size and step."""
        from ..csrc import ops
        found = self._tiles.get(rows_per_tile)
        if found is None:
            tile_cu = torch.empty(self.n_seqs + 1, dtype=torch.int32, device=self.device)
            ops.tile_prefix(self.seq_slot, self.q_len, self.n_seqs, rows_per_tile, tile_cu)
            if self.host is not None:
                bound = sum(-(-q // rows_per_tile) for s, q in zip(self.host.slots, self.host.q_lens) if s >= 0)
            else:
                bound = self.n_seqs * -(-self.max_q_len // rows_per_tile)
            found = self._tiles[rows_per_tile] = (tile_cu, bound)
        return found

    def segments(self, multiple: int = 1, shortest: int = 64, most: int = 16):
        """How a walk over the step's long sequences is cut so that the pieces run side by side: ``(rows per segment,
        prefix sums of segments over the sequences, their bound)``, with segments of at least ``shortest`` rows in
        multiples of ``multiple`` and at most ``most`` for the longest sequence (every segment but a sequence's last
        is walked more than once, so short sequences stay whole); None for steps whose sequences are all short."""
        if self.max_q_len < 2 * shortest:
            return None
        per = -(-self.max_q_len // most)
        seg_rows = max(shortest, -(-per // multiple) * multiple)
        seg_cu, bound = self.tiles(seg_rows)
        return seg_rows, seg_cu, bound

    def kept_zeros(self, shape: tuple[int, ...], dtype: torch.dtype) -> torch.Tensor:
        """A tensor that starts as zeros and lives as long as the context, one per shape and dtype, shared by every
        part that asks: for an output of which a kernel writes only the rows of sequences that take part, while the
        other rows must hold something finite (zeros, or what an earlier step or layer left there) because products
        and norms downstream read whole rows. Cleared once, not once a layer. A part that hands such a tensor on must
        be done with it before the next part of the step asks for the same shape (the parts of a step run one after
        another on one stream, so a mixer's output that the same mixer's projection consumes qualifies)."""
        key = (tuple(shape), dtype)
        found = self._kept.get(key)
        if found is None:
            found = self._kept[key] = torch.zeros(shape, dtype=dtype, device=self.device)
        return found

    def counters(self, n: int) -> torch.Tensor:
        """``n`` int32 zeros for a kernel whose workgroups count themselves: zeros ahead of each launch, and the launch leaves
        zeros. One tensor per length, as old as the context, and apart from ``kept_zeros``, where other things may lie."""
        found = self._counters.get(n)
        if found is None:
            found = self._counters[n] = torch.zeros(n, dtype=torch.int32, device=self.device)
        return found

    def forget_derived(self) -> None:
        """For a context that is used for more than one step: what ``tiles()`` has computed belongs to the step
        before."""
        self._tiles.clear()

    def some_sit_out(self) -> bool:
        """May the step hold sequences that sit out (slot -1)? Without the host's view: yes."""
        return self.host is None or any(s < 0 for s in self.host.slots)


@dataclass
class Partials:
    """A matrix product left as ``count`` float32 partial sums ``[count, rows, width]``."""

    data: torch.Tensor
    count: int

    def summed(self, dtype: torch.dtype) -> torch.Tensor:
        """The product itself, ``[rows, width]``: for a consumer that cannot add the partial sums on its way."""
        from ..csrc import ops
        out = torch.empty(self.data.shape[1:], dtype=dtype, device=self.data.device)
        return ops.sum_partials(self.data, out, self.count)


@dataclass
class Product:
    """A matrix product ``x @ w.T`` not made yet: for a norm that adds it to the residual stream and can have the product's own
    kernel do that. ``made`` makes it as the part that left it would have."""

    x: torch.Tensor
    w: torch.Tensor

    def made(self):
        from .linear import linear
        return linear(self.x, self.w, allow_partials=True)


@dataclass
class LateNormed:
    """Rows ahead of a norm, which the product that reads them takes them through: ``squares`` are float sums of their squares
    (``[count, 8]``), ``weight`` and ``eps`` the norm's."""

    rows: torch.Tensor
    squares: torch.Tensor
    eps: float
    weight: torch.Tensor

    @property
    def late(self) -> tuple:
        return self.squares, self.eps, self.weight


@dataclass
class Deferred:
    """What has still to be added to a float32 residual stream before the next norm reads it, so that one kernel
    can do all of it: a branch's output ``delta`` (a tensor or ``Partials``) that is normed with ``norm`` first (None:
    added as it is), a tensor ``rows`` in the activation dtype that is added row by row (the embedding's output coming
    back), and a ``vector`` added to every row. On a stream of several copies, ``route`` says how ``delta`` enters:
    the part that holds the weights with which the copies are mixed and with which each takes the output."""

    delta: Any = None
    norm: Any = None
    rows: torch.Tensor | None = None
    vector: torch.Tensor | None = None
    route: Any = None

    def picked(self, pick) -> "Deferred":
        """The same for a choice of rows; ``pick`` gathers them from a tensor or from partial sums."""
        return Deferred(pick(self.delta), self.norm, pick(self.rows), self.vector, self.route)


class Part:
    """Base of all parts. ``tensor_specs`` maps logical names to (shape, role, init)."""

    compute_dtype: torch.dtype | None = None    # the dtype the model computes in, set by the model that builds the part

    def tensor_specs(self) -> dict[str, tuple[tuple[int, ...], str, str]]:
        return {}

    def load(self, tensors: dict[str, torch.Tensor]) -> None:
        """Receives the tensors named by ``tensor_specs`` (on the device, in their held dtype)."""

    def kernel_modules(self, dtype: torch.dtype) -> tuple[str, ...]:
        """The kernel libraries this part will call, so they can be compiled together up front."""
        return ()

    # ---- what a step costs, for measurement (rooflines); nothing on the compute path reads these
    def reads_whole(self) -> bool:
        """Does a step read all of this part's tensors (a matrix product does; a row gather does not)?"""
        return True

    def flops(self, rows: int, spans: list[tuple[int, int]]) -> float:
        """Floating-point operations of one step of ``rows`` rows, whose sequences each bring ``q`` rows after
        ``start`` cached ones (``spans`` holds ``(start, q)``): by default two per row and matrix element."""
        if not self.reads_whole():
            return 0.0
        elements = sum(_numel(shape) for shape, role, _ in self.tensor_specs().values() if role == MATRIX)
        return 2.0 * rows * elements


class Norm(Part):
    def forward(self, x: torch.Tensor) -> torch.Tensor:
        raise NotImplementedError

    def add_forward(self, res: torch.Tensor, delta) -> tuple[torch.Tensor, torch.Tensor]:
        """``(res + delta, norm(res + delta))``; ``delta`` is a tensor like ``res`` or ``Partials``."""
        raise NotImplementedError


class Mixer(Part):
    """Mixes information across positions of a sequence; owns the cache line of each of its runs."""

    def cache_need(self):
        """What a run of this mixer keeps per sequence: a ``KVNeed``, a ``StateNeed``, None, or a dictionary from
        names of its own choosing to needs when it keeps several things (keys and values beside fixed-size state,
        two sets of keys with different windows)."""
        return None

    def forward(self, h: torch.Tensor, ctx: StepContext, line, writes_cache: bool):
        """``h`` is ``[rows, hidden]``; returns a tensor of the same shape or ``Partials``. ``line`` is the storage
        ``cache_need`` asked for: a ``KVLine``, a ``StateLine``, None, or a dictionary of those under the same names.
        One that also takes ``leave_product`` may then return a ``Product``."""
        raise NotImplementedError

    def takes_late(self, rows: int, ctx: StepContext) -> bool:
        """Of one that takes ``leave_product``: may the rows of such a step come as ``LateNormed``?"""
        return False

    def left_flops(self, rows: int, positions: dict[str, Any]) -> float:
        """Floating-point operations of the product that ``forward`` leaves unmade where it may, under the model's position
        encodings."""
        return 0.0

    def forward_split(self, h: torch.Tensor, ctx: StepContext, line, writes_cache: bool):
        """``(output without its last bias, that bias or None)``: for a consumer that adds the bias on its own way in
        (a float32 vector of the output's width)."""
        return self.forward(h, ctx, line, writes_cache), None

    def first_products(self, ctx: StepContext) -> list:
        """The products of ``h`` that the mixer begins with, ``(w, out dtype or None)``, where ``forward`` and ``forward_split``
        take them ``made``: for a caller that makes several mixers' together. Empty: none such."""
        return []


class FeedForward(Part):
    row_wise = False    # does a row's output depend on that row of ``h`` alone, and on nothing that ``ctx`` says of the rows?

    def forward(self, h: torch.Tensor, ctx: StepContext):
        raise NotImplementedError

    def takes_late(self, rows: int, ctx: StepContext) -> bool:
        """Of one that takes ``leave_product``: may the rows of such a step come as ``LateNormed``?"""
        return False


def _parameters(function) -> frozenset[str]:
    try:
        return frozenset(inspect.signature(function, follow_wrapped=False).parameters)
    except (TypeError, ValueError):                           # a callable that does not say
        return frozenset()


_parameters_of_methods = functools.lru_cache(maxsize=256)(_parameters)


def accepts(owner, method: str, name: str) -> bool:
    """Does a part's or block's method take the argument ``name``, by its own signature? Asked at every call, since a call may
    be replaced on the object at any time (what a class's method takes is looked up once)."""
    own = vars(owner).get(method)
    return name in (_parameters_of_methods(getattr(type(owner), method)) if own is None else _parameters(own))


def works_row_by_row(ffn) -> bool:
    """``row_wise``, as said by whoever brings the ``forward`` that runs, the object or a class (one that replaces ``forward`` has
    to say it again)."""
    if "forward" in vars(ffn):
        return bool(vars(ffn).get("row_wise", False))
    for cls in type(ffn).__mro__:
        if "row_wise" in vars(cls):
            return bool(ffn.row_wise)
        if "forward" in vars(cls):
            return False
    return False


class StreamPart(Part):
    """Acts on the residual stream between two runs of the schedule (where a pass over a run of layers begins, say):
    a run that names it hands over what is still to be added to the stream and gets back what is to be added now."""

    def enter(self, pending, index: int, ctx: StepContext):
        """``pending`` is what the run before left (None, a tensor, ``Partials`` or ``Deferred``); ``index`` is the
        number the schedule gives this entry. Returns the new pending."""
        raise NotImplementedError


class PositionEncoding(Part):
    def prepare(self, n_positions: int, dtype: torch.dtype, device) -> None:
        """Build whatever tables are needed for positions ``0..n_positions-1``."""


def _numel(shape) -> int:
    n = 1
    for d in shape:
        n *= int(d)
    return n


def matrix(shape) -> tuple[tuple[int, ...], str, str]:
    return (tuple(shape), MATRIX, "normal")
