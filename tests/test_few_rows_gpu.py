"""The experts' products of few rows and the gate/up product of few rows and outputs, alone: at the edges of their tiles,
runs and waves, against float64 arithmetic."""

import math

import pytest
import torch

from test_kernels_gpu import close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ops():
    from dryft_amd.csrc import ops as o
    return o


def within_sums(got, x, w, what):
    """Sums of products of random signs in 32 bits. Added one after the other, partial sum j is some sqrt(j) products large and
    is rounded by some 0.4 x 2^-24 of itself, all of them together by 0.3 x 2^-24 |x| |w|: 3.5 of these units are the largest of
    10^5 sums."""
    want = x.double() @ w.double().T
    most = 5 * 2.0 ** -24 * x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None, :]
    off = (got.cpu().double() - want).abs()
    assert torch.isfinite(got).all() and (off <= most).all(), f"{what}: {float((off / most).max())} of what sums allow"


@pytest.mark.parametrize("rows,experts,top,inter,hidden", [(1, 16, 4, 512, 2048), (4, 16, 4, 520, 1096), (16, 3, 2, 24, 72),
                                                           (16, 1, 1, 8, 64), (2, 40, 7, 33, 1024)])
def test_expert_products_of_few_rows(rows, experts, top, inter, hidden):
    """Gated and plain products: outputs beyond the last group of 16, K that leaves waves without work, tiles of one to
    sixteen places. The unit is computed from sums that are rounded to bfloat16 first, as the kernel's are."""
    o = ops()
    gen = torch.Generator().manual_seed(rows + inter)
    x = torch.randn(rows, hidden, generator=gen).to(torch.bfloat16)
    gate_up = (torch.randn(experts, 2 * inter, hidden, generator=gen) / math.sqrt(hidden)).to(torch.bfloat16)
    chosen = torch.stack([torch.randperm(experts, generator=gen)[:top] for _ in range(rows)]).to(torch.int32)
    plan = o.moe_plan(chosen.to(DEV), experts)
    act = torch.full((rows * top, inter), float("nan"), dtype=torch.bfloat16, device=DEV)
    o.moe_products(x.to(DEV), gate_up.to(DEV), plan, act, top, glu=(float("inf"), 1.0, 0.0))
    place = plan.place_of.cpu().long()
    experts_of = chosen.reshape(-1).long()
    gu = torch.stack([x[p // top].double() @ gate_up[e].double().T for p, e in enumerate(experts_of.tolist())])
    gu = gu.to(torch.bfloat16).double()
    want = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    close(act.cpu()[place], want, torch.bfloat16, ulps=4.0, what="experts' gated products")   # a rounding of each factor, and its own
    down_k = inter // 8 * 8                                               # rows of 16-byte pieces
    if down_k:
        down = torch.randn(experts, hidden, down_k, generator=gen).to(torch.bfloat16)
        a = torch.randn(rows * top, down_k, generator=gen).to(torch.bfloat16)
        y = torch.full((rows * top, hidden), float("nan"), device=DEV)
        o.moe_products(a.to(DEV), down.to(DEV), plan, y, 0)
        for p, e in enumerate(experts_of.tolist()):
            at = place[p]
            within_sums(y[at:at + 1], a[at:at + 1].float(), down[e].float(), "experts' plain products")


@pytest.mark.parametrize("m,inter,k", [(1, 1024, 2048), (8, 3072, 1024), (16, 512, 2048), (3, 9, 8), (16, 37, 1096), (5, 1, 64),
                                       (2, 100, 4104)])
@pytest.mark.parametrize("unit", ["silu", "relu", "clamped"])
def test_gate_up_of_few_rows(m, inter, k, unit):
    torch.manual_seed(m + inter + k)
    x = torch.randn(m, k).to(torch.bfloat16)
    w = (torch.randn(2 * inter, k) * 2 / math.sqrt(k)).to(torch.bfloat16)
    gu = x.double() @ w.double().T
    if unit == "silu":                                          # the unfused path rounds the product and silu first
        gu = gu.to(torch.bfloat16).double()
        want = torch.nn.functional.silu(gu[:, :inter]).to(torch.bfloat16).double() * gu[:, inter:]
    elif unit == "relu":
        want = gu[:, :inter].clamp(min=0) * gu[:, inter:]
    else:
        g, u = gu[:, :inter].clamp(max=1.5), gu[:, inter:].clamp(-1.5, 1.5)
        want = g * torch.sigmoid(1.702 * g) * (u + 1)
    out = ops().gemm_few_glu_bf16(x.to(DEV), w.to(DEV), torch.full((m, inter), float("nan"), dtype=torch.bfloat16, device=DEV),
                                  clamped=(1.5, 1.702) if unit == "clamped" else None, relu=unit == "relu")
    close(out, want, torch.bfloat16, ulps=4.0, what=f"few rows' gated product, {unit}")     # a rounding of each factor, and its own
