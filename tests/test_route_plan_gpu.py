"""Route and plan of a step of few rows in one launch, and the rows and pairs from which they are two."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def check_plan(plan, chosen, experts):
    flat = chosen.flatten().cpu().tolist()
    place_of, sorted_pair, tiles = plan.place_of.cpu().tolist(), plan.sorted_pair.cpu().tolist(), plan.tiles.cpu().tolist()
    n_tiles = int(plan.n_tiles)
    assert sorted(place_of) == list(range(len(flat))) and all(sorted_pair[p] == i for i, p in enumerate(place_of))
    covered = []
    for e, start, count in list(zip(*tiles))[:n_tiles]:
        assert 0 <= e < experts and 1 <= count <= 64
        covered += [(flat[sorted_pair[p]], e) for p in range(start, start + count)]
    assert all(a == b for a, b in covered) and len(covered) == sum(0 <= e < experts for e in flat)


@pytest.mark.parametrize("experts,top", [(1, 1), (8, 2), (16, 4), (64, 8), (64, 64), (65, 3), (130, 5), (512, 4)])
def test_route_and_plan(experts, top):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(experts + top)
    for rows in (1, 2, 7, 16, 17, 40):
        logits = torch.randn(rows, experts + 3, generator=g)
        logits[0, :experts] = logits[0, 0]                                      # ties go to the lower expert
        if rows > 2:
            logits[2, 0] = float("nan")                                         # no number: never chosen while others are left
            logits[1, :experts] = -float("inf")
        chosen, weights = torch.empty((rows, top), dtype=torch.int32, device=DEV), torch.empty((rows, top), device=DEV)
        plan = ops.MoePlan(rows * top, experts, chosen.device, most_places=rows)
        ops.moe_route(logits.to(DEV), None, experts, 1, 1, 1.5, chosen, weights, plan=plan)
        assert plan.done == (rows <= 16 and rows * top <= 64)
        check_plan(plan, chosen, experts)
        for r in range(rows):
            if (rows > 2 and r == 2 and top == experts):
                continue                                                        # nothing but the missing number is left
            s = 1 / (1 + torch.exp(-logits[r, :experts]))
            want = sorted(range(experts), key=lambda e: (-1.0 if s[e].isnan() else -float(s[e]) - 2, e))[:top]
            if not (s[want].diff().abs() < 1e-6).logical_and(s[want].diff() != 0).any():
                assert chosen[r].tolist() == want, (rows, r)
            w = s[chosen[r].cpu().long()]
            assert torch.allclose(weights[r].cpu(), w / (w.sum() + 1e-20) * 1.5, rtol=1e-5, atol=1e-7)
        again = ops.moe_plan(chosen, experts)
        check_plan(again, chosen, experts)
        table = torch.randint(-1, experts + 1, (50, top), generator=g, dtype=torch.int32)
        tokens = torch.randint(0, 50, (rows,), generator=g, dtype=torch.int32)
        plan = ops.MoePlan(rows * top, experts, chosen.device, most_places=rows)
        ops.moe_table_route(tokens.to(DEV), table.to(DEV), experts, chosen, weights, plan=plan)
        assert torch.equal(chosen.cpu(), table[tokens.long()].clamp(0, experts - 1)) and bool((weights == 1 / top).all())
        check_plan(plan, chosen, experts)


@pytest.mark.parametrize("kind", ["sigmoid", "softmax", "chosen_softmax"])
@pytest.mark.parametrize("experts,top,rows", [(1, 1, 3), (16, 4, 4), (16, 4, 40), (64, 8, 9), (130, 5, 7), (130, 5, 40), (512, 4, 33)])
def test_a_row_without_a_number(kind, experts, top, rows):
    """A row whose scores are no numbers (with softmax one logit does that) names experts that exist, its output is no number,
    and the other rows' experts, weights and outputs are what they are beside a row of numbers."""
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(experts + rows)
    good = torch.randn(rows, experts, generator=g)
    bad = good.clone()
    if kind == "softmax":
        bad[1, experts // 2] = float("nan")
    else:
        bad[1] = float("nan")
    x, w = torch.randn(rows, 64, generator=g).to(torch.bfloat16).to(DEV), torch.randn(experts, 32, 64, generator=g).to(torch.bfloat16).to(DEV)

    def run(logits):
        chosen, weights = torch.empty((rows, top), dtype=torch.int32, device=DEV), torch.empty((rows, top), device=DEV)
        plan = ops.MoePlan(rows * top, experts, chosen.device, most_places=rows)
        ops.moe_route(logits.to(DEV), None, experts, 1, 1, 1.0, chosen, weights, softmax=kind == "softmax",
                      chosen_softmax=kind == "chosen_softmax", plan=plan)
        check_plan(plan, chosen, experts)
        y, out = torch.empty((rows * top, 32), device=DEV), torch.empty((rows, 32), dtype=torch.bfloat16, device=DEV)
        ops.moe_products(x, w, plan, y, top)
        ops.moe_combine(y, plan, weights, None, None, 0, out)
        return chosen.cpu(), weights.cpu(), out.cpu()

    want, got = run(good), run(bad)
    others = [r for r in range(rows) if r != 1]
    assert all(torch.equal(a[others], b[others]) for a, b in zip(got, want))
    chosen, weights, out = got
    assert chosen[1].tolist() == list(range(top)) and weights[1].isnan().all() and out[1].isnan().all()


@pytest.mark.parametrize("rows", [5, 40])
def test_plan_of_pairs_without_an_expert(rows):
    """Entries that name no expert get a place behind all others, at any number of pairs."""
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(rows)
    chosen = torch.randint(0, 9, (rows, 3), generator=g, dtype=torch.int32)
    chosen[1, 0], chosen[2], chosen[4, 1] = 9, -1, 0x7fffffff
    plan = ops.moe_plan(chosen.to(DEV), 9)
    check_plan(plan, chosen, 9)
    places = plan.place_of.cpu().view(rows, 3)
    assert sorted(places[(chosen < 0) | (chosen >= 9)].tolist()) == list(range(3 * rows - 5, 3 * rows))
