"""The gate/up product with its activation for many rows, alone: at the edges of its tiles and of its ring of steps."""

import math

import pytest
import torch

from test_kernels_gpu import close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m,inter,k", [(257, 128, 64), (300, 130, 128), (1, 64, 192), (511, 200, 256), (512, 9, 320), (777, 1027, 1024)])
@pytest.mark.parametrize("unit", ["silu", "relu", "clamped"])
def test_gate_up_of_many_rows(m, inter, k, unit):
    from dryft_amd.csrc import ops
    torch.manual_seed(m + inter + k)
    x = torch.randn(m, k + 8).to(torch.bfloat16)                # rows that are not contiguous
    w = (torch.randn(2 * inter, k) * 2 / math.sqrt(k)).to(torch.bfloat16)
    gu = x[:, :k].double() @ w.double().T
    if unit == "silu":                                          # the unfused path rounds the product and silu first
        gu = gu.to(torch.bfloat16).double()
        want = torch.nn.functional.silu(gu[:, :inter]).to(torch.bfloat16).double() * gu[:, inter:]
    elif unit == "relu":
        want = gu[:, :inter].clamp(min=0) * gu[:, inter:]
    else:
        g, u = gu[:, :inter].clamp(max=1.5), gu[:, inter:].clamp(-1.5, 1.5)
        want = g * torch.sigmoid(1.702 * g) * (u + 1)
    out = ops.gemm_many_glu_bf16(x.to(DEV)[:, :k], w.to(DEV), torch.full((m, inter), float("nan"), dtype=torch.bfloat16, device=DEV),
                                 clamped=(1.5, 1.702) if unit == "clamped" else None, relu=unit == "relu")
    close(out, want, torch.bfloat16, ulps=4.0, what=f"many rows' gated product, {unit}")     # a rounding of each factor, and its own
