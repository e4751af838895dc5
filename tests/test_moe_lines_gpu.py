"""Experts' products of few rows, with a shared expert in the same launch: at the edges of their tiles, passes and blocks of K."""

import math

import pytest
import torch

from test_kernels_gpu import close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def unit_of(z, kind):
    """The unit in 64 bits on a product's rounded results."""
    z = z.to(torch.bfloat16).double()
    if kind == "relu2":
        return z.clamp(min=0) ** 2
    g, u = z[:, :z.shape[1] // 2], z[:, z.shape[1] // 2:]
    if kind == "silu":
        return torch.nn.functional.silu(g) * u
    g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
    return g * torch.sigmoid(1.702 * g) * (u + 1)


@pytest.mark.parametrize("rows,experts,top", [(1, 4, 4), (3, 5, 2), (4, 16, 4), (5, 3, 3), (8, 2, 1), (9, 2, 1), (16, 1, 1), (16, 16, 4)])
@pytest.mark.parametrize("k,inter,shared_inter", [(8, 8, 16), (136, 24, 72), (512, 72, 8), (1160, 136, 200)])
@pytest.mark.parametrize("kind", ["silu", "clamped", "relu2"])
def test_experts_and_the_shared_one(rows, experts, top, k, inter, shared_inter, kind):
    from dryft_amd.csrc import ops
    torch.manual_seed(rows * 1000 + k + inter)
    halves = 1 if kind == "relu2" else 2
    x = torch.randn(rows, k + 8).to(torch.bfloat16)[:, :k]                     # rows wider apart than K
    w = (torch.randn(experts, halves * inter, k) * 2 / math.sqrt(k)).to(torch.bfloat16)
    down = (torch.randn(experts, k, inter) / math.sqrt(inter)).to(torch.bfloat16)
    ws = (torch.randn(halves * shared_inter, k) * 2 / math.sqrt(k)).to(torch.bfloat16)
    down_s = (torch.randn(k, shared_inter) / math.sqrt(shared_inter)).to(torch.bfloat16)
    chosen = torch.stack([torch.randperm(experts)[:top] for _ in range(rows)]).to(torch.int32)
    plan = ops.moe_plan(chosen.to(DEV), experts)
    n = rows * top
    act, y = torch.full((n, inter), float("nan"), dtype=torch.bfloat16, device=DEV), torch.full((n, k), float("nan"), device=DEV)
    act_s = torch.full((rows, shared_inter), float("nan"), dtype=torch.bfloat16, device=DEV)
    y_s = torch.full((rows, k), float("nan"), dtype=torch.bfloat16, device=DEV)
    how = dict(act="relu2") if kind == "relu2" else dict(glu=(float("inf"), 1.0, 0.0) if kind == "silu" else (1.5, 1.702))
    ride = (x.to(DEV) if x.is_contiguous() else torch.nn.functional.pad(x, (0, 8)).to(DEV)[:, :k], ws.to(DEV), act_s,
            (1.5, 1.702) if kind == "clamped" else None)
    ops.moe_products(ride[0], w.to(DEV), plan, act, top, shared=ride, **how)
    ops.moe_products(act, down.to(DEV), plan, y, 0, shared=(act_s, down_s.to(DEV), y_s, None))
    place = plan.place_of.cpu().view(rows, top)
    a = act.cpu().double()
    for r in range(rows):
        for t in range(top):
            e, p = int(chosen[r, t]), int(place[r, t])
            # the unit's argument is a bfloat16 step off where its sum lies between two
            close(act[p:p + 1], unit_of(x[r:r + 1].double() @ w[e].double().T, kind), torch.bfloat16, ulps=4.0, what=f"row {r} expert {e}")
            close(y[p:p + 1], a[p:p + 1] @ down[e].double().T, torch.float32, what=f"row {r} expert {e}, back")
    close(act_s, unit_of(x.double() @ ws.double().T, kind), torch.bfloat16, ulps=4.0, what="shared")
    close(y_s, act_s.cpu().double() @ down_s.double().T, torch.bfloat16, what="shared, back")


@pytest.mark.parametrize("rows,experts,top", [(1, 4, 4), (4, 16, 2), (6, 3, 3), (9, 2, 2), (16, 1, 1), (16, 16, 4)])
@pytest.mark.parametrize("k,inter", [(64, 24), (248, 1024), (256, 520), (512, 72), (1032, 512), (1024, 1080)])
@pytest.mark.parametrize("kind", ["silu", "clamped", "relu2"])
def test_experts_alone(rows, experts, top, k, inter, kind):
    """Without a shared expert the kernel follows from rows, places and K: every one it may be, on both sides of the lines."""
    from dryft_amd.csrc import ops
    torch.manual_seed(rows * 1000 + k + inter)
    halves = 1 if kind == "relu2" else 2
    x = torch.randn(rows, k).to(torch.bfloat16)
    w = (torch.randn(experts, halves * inter, k) * 2 / math.sqrt(k)).to(torch.bfloat16)
    down = (torch.randn(experts, k, inter) / math.sqrt(inter)).to(torch.bfloat16)
    chosen = torch.stack([torch.randperm(experts)[:top] for _ in range(rows)]).to(torch.int32)
    plan = ops.moe_plan(chosen.to(DEV), experts)
    act, y = torch.full((rows * top, inter), float("nan"), dtype=torch.bfloat16, device=DEV), torch.full((rows * top, k), float("nan"), device=DEV)
    how = dict(act="relu2") if kind == "relu2" else dict(glu=(float("inf"), 1.0, 0.0) if kind == "silu" else (1.5, 1.702))
    ops.moe_products(x.to(DEV), w.to(DEV), plan, act, top, **how)
    ops.moe_products(act, down.to(DEV), plan, y, 0)
    place = plan.place_of.cpu().view(rows, top)
    a = act.cpu().double()
    for e in range(experts):
        at = [(r, int(place[r, t])) for r in range(rows) for t in range(top) if int(chosen[r, t]) == e]
        if at:
            r, p = [i for i, _ in at], [j for _, j in at]
            close(act[p], unit_of(x[r].double() @ w[e].double().T, kind), torch.bfloat16, ulps=4.0, what=f"expert {e}")
            close(y[p], a[p] @ down[e].double().T, torch.float32, what=f"expert {e}, back")


@pytest.mark.parametrize("unit", ["silu", "clamped", "relu2"])
@pytest.mark.parametrize("how", ["object", "class", "exchanged"])
def test_a_replaced_shared_expert_is_called(monkeypatch, unit, how):
    """A shared expert whose ``forward`` was replaced, or that is another part, adds what it says to what the routed ones give without one."""
    from dryft_amd.csrc import ops
    from dryft_amd.parts.base import FeedForward
    from dryft_amd.parts.experts import RoutedExperts
    torch.manual_seed(0)
    make = lambda shared: RoutedExperts(64, 4, 2, 64, limit=1.5 if unit == "clamped" else None, unit=unit, shared=shared, correction=False, shared_gate=False)
    part, alone = make((24, 1.5)), make(None)
    part.compute_dtype = alone.compute_dtype = torch.bfloat16
    tensors = {name: torch.randn(*spec[0]).to(torch.bfloat16).to(DEV) * 0.1 for name, spec in part.tensor_specs().items()}
    part.load(tensors)
    alone.load(tensors)
    h, plan = torch.randn(3, 64).to(torch.bfloat16).to(DEV), ops.MoePlan(6, 4, DEV, most_places=3)
    assert part._shared_rides(h, plan)
    half = lambda *a, **k: torch.full((3, 64), 0.5, dtype=torch.bfloat16, device=DEV)
    if how == "object":
        part.shared.forward = half
    elif how == "class":
        monkeypatch.setattr(type(part.shared), "forward", half)
    else:
        part.shared = type("Half", (FeedForward,), {"forward": half})()
    # both sides round the routed sum once to bfloat16, one of them with 0.5 added
    got, want = part.forward(h, None).double(), alone.forward(h, None).double() + 0.5
    assert bool(((got - want).abs() <= 2.0 ** -8 * (got.abs() + (want - 0.5).abs())).all())
