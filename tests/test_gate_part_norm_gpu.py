"""The state-space read-out's gate and norm by parts, eight values a thread: parts of one run and of several a thread, parts that do not
fill a wave, rows that sit out, and widths and columns that the plain kernel takes, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("inner,parts,col", [(2048, 2, 8), (8, 1, 0), (24, 3, 16), (4096, 1, 0), (8192, 1, 8), (1040, 2, 0), (8200, 1, 8), (30, 3, 4), (64, 2, 3)])
def test_gate_part_norm(dtype, inner, parts, col):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(inner + parts)
    rows, eps = 5, 1e-5
    y, w = torch.randn(rows, inner, generator=g), torch.randn(inner, generator=g)
    z = torch.randn(rows, -(-(inner + col) // 8) * 8, generator=g).to(dtype)
    slots = torch.tensor([3, -1, 0, 7, 1], dtype=torch.int32)
    out = torch.full((rows, inner), 7.0, dtype=dtype, device=DEV)
    ops.gate_part_norm(y.to(DEV), z.to(DEV), col, w.to(DEV), slots.to(DEV), out, parts, eps)
    v = (y.double() * torch.nn.functional.silu(z[:, col:col + inner].double())).view(rows, parts, -1)
    want = (v * (v.pow(2).mean(-1, keepdim=True) + eps).rsqrt()).view(rows, inner) * w.double()
    got, live = out.double().cpu(), slots >= 0
    # a float sum of up to 8,200 squares in parts of a wave, and a few roundings more; bfloat16 rounds the result once
    tol = 32 * 2.0 ** -24 * want.abs() + 1e-6 + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0.0)
    assert not got[~live].any() and bool(((got - want).abs() <= tol)[live].all())
