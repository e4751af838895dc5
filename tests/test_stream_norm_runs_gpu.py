"""The norms of a residual stream whose rows stay in registers: widths at the edges of one, two and four runs a thread
(512 threads x 8 values), more parts than are asked for at once, parts of a row, and a misaligned row."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-5
# float32: sums of up to 16,384 squares added in a tree and a reciprocal root, a few 2^-24 each; bfloat16: one rounding, 2^-9.
TOL = {torch.float32: 2e-6, torch.bfloat16: 2 ** -8}


def normed(x, w, centred, groups):
    x = x.view(x.shape[0], groups, -1)
    if centred:
        x = x - x.mean(-1, keepdim=True)
    return (x / (x.pow(2).mean(-1, keepdim=True) + EPS).sqrt()).flatten(1) * w


def close(got, want, tol):
    got = got.double().cpu()
    assert torch.isfinite(got).all()
    assert float((got - want).abs().max() / want.abs().max()) <= tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,parts,groups", [(8, 1, 1), (504, 9, 1), (4096, 8, 4), (4104, 11, 1), (8192, 3, 256),
                                                (8200, 2, 25), (16384, 1, 2), (12296, 17, 1)])
def test_stream_norm_runs(dtype, width, parts, groups):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(width + parts)
    rows = 3
    x = torch.randn(rows, width, generator=g) + 0.5
    d = torch.randn(parts, rows, width, generator=g)
    wb, w, b = (torch.randn(width, generator=g) for _ in range(3))
    for centred in (False, True) if groups == 1 else (False,):
        for delta in ((d.to(DEV), parts), d[0].to(dtype).to(DEV)):
            dd = d.double().sum(0) if isinstance(delta, tuple) else d[0].to(dtype).double()
            x_dev, y = x.clone().to(DEV), torch.empty(rows, width, dtype=dtype, device=DEV)
            ops.stream_norm(x_dev, delta, wb.to(DEV), None, None, w.to(DEV), EPS, x_dev, y, dtype, groups=groups,
                            centred=centred, post_centred=centred, bias=b.to(DEV) if groups == 1 else None)
            want = x.double() + normed(dd, wb.double(), centred, 1)
            close(x_dev, want, 2e-6)
            close(y, normed(want, w.double(), centred, groups) + (b.double() if groups == 1 else 0), TOL[dtype])
    # one value off 16 bytes: the same row by the other kernel
    y1, y2 = (torch.empty(rows, width, dtype=dtype, device=DEV) for _ in range(2))
    off = torch.empty(rows * width + 1, device=DEV)[1:].view(rows, width).copy_(x)
    for src, y in ((x.to(DEV), y1), (off, y2)):
        ops.stream_norm(src, None, None, None, None, w.to(DEV), EPS, None, y, dtype, groups=groups)
    close(y2, y1.double().cpu(), TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,groups", [(2040, 8), (72, 8), (3000, 24), (40, 10), (504, 56), (4104, 36), (8200, 8), (12296, 8),
                                          (16376, 8)])
def test_parts_that_end_within_a_run(dtype, width, groups):
    """Parts whose length is no multiple of 8: runs of eight values that reach into the next part, once and twice in a row."""
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(width)
    x, w = torch.randn(3, width, generator=g) * torch.linspace(0.1, 3, width), torch.randn(width, generator=g)
    d = torch.randn(2, 3, width, generator=g)
    x_out, y = torch.empty(3, width, device=DEV), torch.empty(3, width, dtype=dtype, device=DEV)
    ops.stream_norm(x.to(DEV), (d.to(DEV), 2), None, None, None, w.to(DEV), EPS, x_out, y, dtype, groups=groups)
    want = x.double() + d.double().sum(0)
    close(x_out, want, 2e-6)
    close(y, normed(want, w.double(), False, groups), TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,parts", [(8, 1), (520, 9), (4096, 8), (4104, 3), (8192, 12)])
def test_pair_mean_runs(dtype, width, parts):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(width)
    a = torch.randn(3, width, generator=g).to(dtype)
    b = 0.1 * torch.randn(parts, 3, width, generator=g)
    bias, wa, wb = (torch.randn(width, generator=g) for _ in range(3))
    out = torch.empty(3, width, device=DEV)
    want = 0.5 * (normed(a.double() + bias.double(), wa.double(), False, 1) + normed(b.double().sum(0), wb.double(), False, 1))
    ops.rms_pair_mean(a.to(DEV), bias.to(DEV), wa.to(DEV), (b.to(DEV), parts), None, wb.to(DEV), EPS, out, dtype)
    close(out, want, 2e-6)
    ops.rms_pair_mean((b.to(DEV), parts), None, wb.to(DEV), a.to(DEV), bias.to(DEV), wa.to(DEV), EPS, out, dtype)
    close(out, want, 2e-6)
