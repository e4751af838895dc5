"""Products of 17 to 128 rows whose operands go straight into LDS, at the edges of their tiles of rows and of outputs."""

import math

import pytest
import torch

from test_kernels_gpu import close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m", [5, 17, 64, 65, 80, 81, 96])
@pytest.mark.parametrize("inter,k,waves", [(47, 128, 0), (100, 640, 5), (136, 256, 8), (1024, 2560, 4), (6152, 2048, 0)])
@pytest.mark.parametrize("unit", ["silu", "relu", "clamped"])
def test_panel_of_up_to_96_rows(m, inter, k, waves, unit):
    """One to six tiles of rows, three stages in LDS and (eight waves at 96 rows) two; weights kept and, from 48 MiB on, read once; rows of
    x wider apart than K."""
    from dryft_amd.csrc import ops
    torch.manual_seed(m + inter + k)
    x = torch.randn(m, k + 8).to(torch.bfloat16)
    w = (torch.randn(2 * inter, k) * 2 / math.sqrt(k)).to(torch.bfloat16)
    gu = x[:, :k].double() @ w.double().T
    if unit == "silu":                                          # the product and silu are rounded first
        gu = gu.to(torch.bfloat16).double()
        want = torch.nn.functional.silu(gu[:, :inter]).to(torch.bfloat16).double() * gu[:, inter:]
    elif unit == "relu":
        want = gu[:, :inter].clamp(min=0) * gu[:, inter:]
    else:
        g, u = gu[:, :inter].clamp(max=1.5), gu[:, inter:].clamp(-1.5, 1.5)
        want = g * torch.sigmoid(1.702 * g) * (u + 1)
    out = torch.full((m, inter), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.gemm_panel_swiglu_bf16(x.to(DEV)[:, :k], w.to(DEV), out, waves, (1.5, 1.702) if unit == "clamped" else None, unit == "relu")
    close(out, want, torch.bfloat16, ulps=4.0, what=f"panel, {unit}")        # a rounding of each factor, and its own


@pytest.mark.parametrize("m", [17, 33, 64, 65, 81, 97, 128])
@pytest.mark.parametrize("n,k,waves,splits", [(77, 64, 5, 1), (97, 320, 6, 5), (100, 192, 8, 3), (2560, 1664, 5, 7),
                                              (33000, 128, 8, 1), (20500, 192, 4, 1), (4200, 1024, 4, 4), (2056, 2048, 8, 16),
                                              (2560, 9728, 5, 8), (6144, 2560, 6, 4), (33000, 1024, 8, 1), (1531, 2560, 8, 2),
                                              (1200, 1280, 5, 1), (1000, 1600, 6, 1), (25000, 832, 6, 1), (7000, 3072, 8, 4)])
def test_products_of_17_to_128_rows(m, n, k, waves, splits):
    """Every width of a workgroup, runs of K of one group and of unequal length, weights kept and read once, launches of more
    workgroups than compute units (two stages in LDS); a row of x wider than K. And runs several times as long as the ring of two to four
    stages, in each of these: what a wrong wait or stage would show in."""
    from dryft_amd.csrc import ops
    torch.manual_seed(m + n + k)
    x, w = torch.randn(m, k + 8).to(torch.bfloat16).to(DEV)[:, :k], (torch.randn(n, k) / math.sqrt(k)).to(torch.bfloat16).to(DEV)
    assert ops.gemm_mid_splits(k, splits) == splits
    parts = torch.full((splits, m, n), float("nan"), dtype=torch.float32, device=DEV)
    ops.gemm_mid_bf16(x, w, parts, splits, waves)
    per = -(-(k // 64) // splits)
    for s in range(splits):
        a, b = 64 * per * s, min(k, 64 * per * (s + 1))
        close(parts[s], x[:, a:b].double() @ w[:, a:b].double().T, torch.float32, what=f"run {s}")
