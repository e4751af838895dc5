"""Products of at most 16 rows whose loads are matrix-core operands as they are: edges of blocks of K, of a workgroup's rows and of
the groups of four rows of x; the norm between two products without a launch of its own."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def ops():
    from dryft_amd.csrc import ops
    return ops


def operands(m, n, k, seed, stride=0):
    torch.manual_seed(seed)
    x = torch.randn(m, stride or k, device=DEV).to(torch.bfloat16)[:, :k]
    w = (torch.randn(n, k, device=DEV) * k ** -0.5).to(torch.bfloat16)
    return x, w


def product(x, w):
    """In 64 bits, and how far a float sum in any order may be from it: a rounding per addition."""
    x, w = x.double(), w.double()
    return x @ w.T, x.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs().T)


# one, four, five, eight, nine and 16 rows (groups of four); K of one piece, around a block of 128 and past all waves' first blocks;
# outputs around the lines between shapes (1,024, 2,048, 2,560, 3,072) and of 20 rows a workgroup (40 Mi values of W)
CASES = [(1, 1, 8), (4, 3, 24), (5, 4, 120), (3, 5, 128), (8, 1024, 136), (9, 1025, 1032), (16, 2049, 1288), (2, 2561, 72), (7, 3073, 2568),
         (16, 4099, 520), (6, 5123, 8200), (12, 5120, 8192), (1, 3072, 9728)]


@pytest.mark.parametrize("m,n,k", CASES)
def test_product(m, n, k):
    x, w = operands(m, n, k, m + n + k, stride=k + 8)
    want, bound = product(x, w)
    out = ops().gemm_lines_bf16(x, w, torch.full((m, n), float("nan"), device=DEV))
    assert (out.double() - want).abs().le(bound).all()
    rounded = ops().gemm_lines_bf16(x, w, torch.full((m, n), float("nan"), device=DEV).to(torch.bfloat16))
    assert torch.equal(rounded, out.to(torch.bfloat16))


@pytest.mark.parametrize("m,n,k", CASES)
@pytest.mark.parametrize("weights", [torch.bfloat16, torch.float32])
def test_norm_between_products(m, n, k, weights):
    o = ops()
    x, w = operands(m, n, k, m + n + k + 1)
    residual = torch.randn(m, n, device=DEV).to(torch.bfloat16)
    weight = (1 + 0.3 * torch.randn(n, device=DEV)).to(weights)
    before = residual.double()
    want, bound = product(x, w)
    rows, squares = o.gemm_lines_next_bf16(x, w, residual, weight)
    # the sum of the residual and the product, rounded once
    want = before + want
    assert (residual.double() - want).abs().le(2.0 ** -8 * want.abs() + 1.01 * bound).all()
    assert torch.equal(rows, (residual.float() * weight.float()).to(torch.bfloat16))
    total = (residual.double() ** 2).sum(1)
    assert (squares.double().sum(0)[:m] - total).abs().le(n * 2.0 ** -24 * total).all()
    # the product that follows, against the norm by its formula on those rows
    k2 = n // 8 * 8
    if k2 != n or squares.shape[0] > o.LATE_MOST:
        return
    x2, w2 = rows, operands(1, 40, n, 5)[1]
    want, bound = product(x2, w2)
    scale = torch.rsqrt(total / n + 1e-6)[:, None]
    out = o.gemm_lines_bf16(x2, w2, torch.empty((m, 40), device=DEV), late=(squares, 1e-6))
    slack = (n + 8) * 2.0 ** -24                                # of the squares' sums and of the root
    assert (out.double() - want * scale).abs().le((bound + slack * want.abs()) * scale * 1.01).all()


@pytest.mark.parametrize("m,inter,k", [(3, 1024, 256), (8, 1025, 2560), (16, 30, 1024)])
def test_gate_up_after_a_norm(m, inter, k):
    """Scaling the sums is scaling the rows: by powers of two that is exact."""
    o = ops()
    x, w = operands(m, 2 * inter, k, m + inter)
    exponent = torch.arange(m, device=DEV) % 3 - 1
    squares = torch.zeros((300, 16), device=DEV)
    squares[7, :m] = k * 4.0 ** exponent                        # rsqrt(squares / k) = 2 ** -exponent
    got = o.gemm_few_glu_bf16(x, w, torch.empty((m, inter), dtype=torch.bfloat16, device=DEV), late=(squares, 0.0))
    scaled = (x.float() * 2.0 ** -exponent[:, None]).to(torch.bfloat16)
    want = o.gemm_few_glu_bf16(scaled, w, torch.empty((m, inter), dtype=torch.bfloat16, device=DEV))
    close = (got.double() - want.double()).abs().le(2.0 ** -7 * want.double().abs() + 1e-6)
    assert close.all()


def test_refusals():
    o = ops()
    x, w = operands(17, 8, 64, 0)
    with pytest.raises(o.KernelError):
        o.gemm_lines_bf16(x, w, torch.empty((17, 8), device=DEV))
    x, w = operands(2, 8, 60, 0)
    with pytest.raises(o.KernelError):
        o.gemm_lines_bf16(x, w, torch.empty((2, 8), device=DEV))
    x, w = operands(2, 8, 64, 0)
    with pytest.raises(o.KernelError):
        o.gemm_lines_bf16(x, w, torch.empty((2, 8), device=DEV), late=(torch.zeros((1025, 16), device=DEV), 0.0))
