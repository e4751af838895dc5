"""What a block hands to its parts, and a model to its blocks, follows from the calls that are there when it runs."""

import functools
import gc
import types
import weakref

import pytest
import torch

from dryft_amd.parts.base import FeedForward, LateNormed, Mixer, Norm, Product, accepts, works_row_by_row
from dryft_amd.parts.block import PreNormBlock


@pytest.fixture(autouse=True)
def made_here(monkeypatch):
    monkeypatch.setattr(Product, "made", lambda product: product.x @ product.w.T)


class PlainNorm(Norm):
    def forward(self, x):
        return 2 * x

    def add_forward(self, res, delta, late=False):
        self.late = late
        if isinstance(delta, Product):
            if late:
                res = res + delta.x @ delta.w.T
                return res, LateNormed(res, None, 0.0, None)
            delta = delta.x @ delta.w.T
        return res + delta, 2 * (res + delta)


class Leaves:
    def __init__(self):
        self.w = torch.eye(4)

    def end(self, h, leave_product):
        self.seen = h, leave_product
        h = 2 * h.rows if isinstance(h, LateNormed) else h
        return Product(h, self.w) if leave_product else h @ self.w.T


class PlainMixer(Leaves, Mixer):
    def forward(self, h, ctx, line, writes_cache, leave_product=False):
        return self.end(h, leave_product)


class PlainFFN(Leaves, FeedForward):
    row_wise = True

    def forward(self, h, ctx, leave_product=False):
        return self.end(h, leave_product)


class LateFFN(PlainFFN):
    def takes_late(self, rows, ctx):
        return True


CAPTURED, STEP = types.SimpleNamespace(host=None), types.SimpleNamespace(host="the step as the host knows it")


def run(block, rows=2):
    x, pending = block.forward(torch.ones(rows, 4), None, STEP, None, True, leave_product=True)
    return x + (pending.x @ pending.w.T if isinstance(pending, Product) else pending)


def expected(rows):
    mixed = torch.ones(rows, 4) * 3
    return mixed + 2 * mixed


def hooks(call):
    """The ways to put a call in the place of another that takes what every such part takes, and no more."""
    def short(h, ctx):
        return call(h, ctx)

    def passes_on(*args, **kw):
        return call(*args, **kw)

    return [short, passes_on, functools.wraps(call)(short), functools.partial(short), functools.partial(passes_on)]


@pytest.mark.parametrize("which", range(5))
@pytest.mark.parametrize("ffn", [PlainFFN, LateFFN])
def test_a_replaced_feed_forward_gets_plain_rows(which, ffn):
    block = PreNormBlock(PlainNorm(), PlainMixer(), PlainNorm(), ffn())
    assert block.picks_rows and torch.equal(run(block), expected(2)) and block.ffn.seen[1]
    assert isinstance(block.ffn.seen[0], LateNormed) == (ffn is LateFFN)         # one that does not say takes plain rows
    block.ffn.forward = hooks(block.ffn.forward)[which]
    assert torch.equal(run(block), expected(2))
    assert not block.ffn.seen[1] and not isinstance(block.ffn.seen[0], LateNormed)
    assert not block.picks_rows                                                  # it may look at all rows
    block.ffn.row_wise = True
    assert block.picks_rows
    del block.ffn.forward
    assert torch.equal(run(block), expected(2)) and block.ffn.seen[1]


def test_a_replaced_norm_and_an_exchanged_part():
    block = PreNormBlock(PlainNorm(), PlainMixer(), PlainNorm(), LateFFN())
    add = block.ffn_norm.add_forward
    block.ffn_norm.add_forward = lambda res, delta: add(res, delta)
    made = []
    block.mixer.forward = lambda h, ctx, line, writes_cache, call=block.mixer.forward: (made.append(1), call(h, ctx, line, writes_cache))[1]
    assert torch.equal(run(block), expected(2)) and made and not block.ffn_norm.late

    class Other(FeedForward):
        def forward(self, h, ctx):
            return h

    block.ffn = Other()
    assert torch.equal(run(block), expected(2)) and not block.picks_rows


@pytest.mark.parametrize("rows,ctx,left", [(1, STEP, True), (8, STEP, True), (9, STEP, False), (300, STEP, False), (8, CAPTURED, True),
                                           (256, CAPTURED, True), (257, CAPTURED, False)])
def test_products_of_many_rows_are_made_where_they_stand(rows, ctx, left):
    """One left unmade keeps its operand alive until the next layer is through, which a long prompt's are too large for."""
    block = PreNormBlock(PlainNorm(), PlainMixer(), PlainNorm(), PlainFFN())
    x, pending = block.forward(torch.ones(rows, 4), None, ctx, None, True, leave_product=True)
    assert isinstance(pending, Product) == block.mixer.seen[1] == block.ffn.seen[1] == left
    # rows that are picked behind the mixer: its product is then made of those alone
    x, pending = block.forward(torch.ones(rows, 4), None, ctx, None, True, leave_product=True,
                               pick=lambda t: Product(t.x[:1], t.w) if isinstance(t, Product) else t[:1])
    assert block.mixer.seen[1] and x.shape[0] == 1 and isinstance(pending, Product)


def test_replaced_calls_are_not_kept():
    part = PlainFFN()
    part.forward = lambda h, ctx: h
    gone = weakref.ref(part.forward)
    assert not accepts(part, "forward", "leave_product") and accepts(PlainFFN(), "forward", "leave_product")
    del part.forward
    gc.collect()
    assert gone() is None and works_row_by_row(part)


@pytest.mark.parametrize("name", ["forward", "forward_split"])
def test_mixers_side_by_side_with_a_replaced_call_begin_alone(monkeypatch, name):
    """Two mixers' first products are made together only where the calls that run take them."""
    from dryft_amd.parts import parallel

    class Begins(Mixer):
        def first_products(self, ctx):
            return [(torch.eye(4), None)]

        def forward(self, h, ctx, line, writes_cache, made=None):
            self.made = made
            return (made[0] if made else h) * 2

        def forward_split(self, h, ctx, line, writes_cache, made=None):
            return self.forward(h, ctx, line, writes_cache, **({"made": made} if made else {})), None

    monkeypatch.setattr(parallel, "together_pay", lambda h, weights: len(weights) == 2)
    monkeypatch.setattr(parallel, "linears", lambda h, products: [h @ w.T for w, _ in products])
    both = parallel.ParallelMixer.__new__(parallel.ParallelMixer)
    both.mixers = {"left": Begins(), "right": Begins()}
    h = torch.ones(2, 4)
    assert {n: len(m["made"]) for n, m in both._first_products(h, STEP).items()} == {"left": 1, "right": 1}
    if name == "forward":
        both.mixers["left"].forward = lambda h, ctx, line, writes_cache: 3 * h
    else:
        both.mixers["left"].forward_split = lambda h, ctx, line, writes_cache: (3 * h, None)
    assert both._first_products(h, STEP) == {}
    assert torch.equal(both.mixers["left"].forward_split(h, STEP, None, True)[0], 3 * h)


def routed(unit):
    from dryft_amd.parts.experts import RoutedExperts
    part = RoutedExperts(64, 4, 2, 64, limit=2.0 if unit == "clamped" else None, unit=unit, shared=(128, 2.0), correction=False)
    part.load({name: torch.zeros(*spec[0], dtype=torch.bfloat16) for name, spec in part.tensor_specs().items()})
    return part


@pytest.mark.parametrize("unit", ["silu", "clamped", "relu2"])
def test_only_the_shared_expert_that_was_made_rides_along(monkeypatch, unit):
    """A shared expert whose call is replaced, on the object or on its class, or that is exchanged for one of another unit, runs as it
    says and not in the routed ones' launches, which know the unit of the routed ones alone."""
    from dryft_amd.csrc import ops
    from dryft_amd.parts.mlp import ClampedGLU, ReGLU, SquaredReLU, SwiGLU
    part, h, plan = routed(unit), torch.zeros(3, 64, dtype=torch.bfloat16), ops.MoePlan(6, 4, "cpu", most_places=3)
    made, own = part.shared, type(part.shared)
    assert part._shared_rides(h, plan)
    made.forward = lambda h, ctx: h
    assert not part._shared_rides(h, plan)
    del made.forward
    with monkeypatch.context() as m:
        m.setattr(own, "forward", lambda self, h, ctx, leave_product=False: h)
        assert not part._shared_rides(h, plan)
    assert part._shared_rides(h, plan)
    for other in (ClampedGLU(64, 128, 2.0), SwiGLU(64, 128), ReGLU(64, 128), SquaredReLU(64, 128)):
        if type(other) is own:
            continue
        other.load({name: torch.zeros(*spec[0], dtype=torch.bfloat16) for name, spec in other.tensor_specs().items()})
        part.shared = other
        assert not part._shared_rides(h, plan), type(other)
    part.shared = made
    if unit == "silu":
        made.relu = True                                     # the gated unit's own switch
        assert not part._shared_rides(h, plan)
