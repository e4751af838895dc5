"""Products of the same few rows in one launch: at the edges of their workgroups, and where two mixers begin side by side."""

import math

import pytest
import torch

from test_kernels_gpu import close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("outputs,k", [((12,), 8), ((1, 1, 1, 1), 136), ((100, 7), 2048), ((2048, 32, 3), 520), ((3100, 12, 13, 500), 264),
                                       ((6, 40000), 64)])
def test_products_beside_one_another(m, outputs, k):
    from dryft_amd.csrc import ops
    torch.manual_seed(m + sum(outputs) + k)
    x = torch.randn(m, k + 8).to(torch.bfloat16).to(DEV)[:, :k]
    products = []
    for i, n in enumerate(outputs):
        w = (torch.randn(n, k) / math.sqrt(k)).to(torch.bfloat16).to(DEV)
        products.append((w, torch.full((m, n), float("nan"), dtype=torch.float32 if i % 2 else torch.bfloat16, device=DEV)))
    ops.gemm_lines_beside(x, products)
    for i, (w, out) in enumerate(products):
        close(out, x.double() @ w.double().T, out.dtype, what=f"product {i}")


def test_products_beside_one_another_refuse():
    from dryft_amd.csrc import ops
    x, w = torch.zeros(17, 64, dtype=torch.bfloat16, device=DEV), torch.zeros(8, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ops.KernelError, match="few rows"):
        ops.gemm_lines_beside(x, [(w, torch.empty(17, 8, device=DEV))])
    with pytest.raises(ops.KernelError, match="1 to 4"):
        ops.gemm_lines_beside(x[:4], [(w, torch.empty(4, 8, device=DEV))] * 5)
    with pytest.raises(ops.KernelError, match="out contiguous"):
        ops.gemm_lines_beside(x[:4], [(w, torch.empty(4, 9, device=DEV))])
