"""The short convolution of many rows, four rows a thread: equal, bit for bit, to a row a thread, over sequences that start, that go on and
that sit out, runs across their starts and rows that are no multiple of four; and against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("channels,taps,col", [(4096, 4, 8), (5440, 3, 0), (8200, 2, 16)])
def test_four_rows_a_thread(dtype, channels, taps, col):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(channels + taps)
    lens, first, slots = [1, 2, 3, 501, 6, 300, 217], [0, 5, 1, 0, 2, 40, 0], [3, 0, 5, 1, -1, 2, 6]
    n = sum(lens)
    assert n * channels * taps >= 16 << 20 and n // 16 >= len(lens) and n % 4
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    seq = [s for s, k in enumerate(lens) for _ in range(k)]
    pos = [p + i for p, k in zip(first, lens) for i in range(k)]
    u = torch.randn(n, channels + col, generator=g).to(dtype).to(DEV)
    w = torch.randn(channels, taps, generator=g).to(DEV)
    ib, ob = torch.randn(channels, generator=g).to(DEV), torch.randn(channels, generator=g).to(DEV)
    tail = torch.randn(7, taps - 1, channels, generator=g).to(DEV)
    facts = ints([slots[s] for s in seq]), ints(seq), ints(pos), ints(first)
    for in_bias, out_bias, silu in ((None, None, False), (ib, ob, True)):
        want, got = (torch.full((n, channels), 9.0, dtype=dtype, device=DEV) for _ in range(2))
        ops.causal_conv(u, col, channels, in_bias, w, out_bias, silu, *facts, tail, want, weight_t=w.t().contiguous(), n_seqs=n)
        ops.causal_conv(u, col, channels, in_bias, w, out_bias, silu, *facts, tail, got, weight_t=w.t().contiguous())
        assert torch.equal(got, want)
        s, at = 3, sum(lens[:3])                     # the sequence that starts, in 64 bits: zeros ahead of it
        x = u[at:at + lens[s], col:].double() + (in_bias.double() if in_bias is not None else 0.0)
        x = torch.nn.functional.pad(x, (0, 0, taps - 1, 0))
        terms = [x[j:j + lens[s]] * w[:, j].double() for j in range(taps)]
        y = sum(terms) + (out_bias.double() if out_bias is not None else 0.0)
        size = sum(t.abs() for t in terms) + (out_bias.double().abs() if out_bias is not None else 0.0)
        y = torch.nn.functional.silu(y) if silu else y
        # a rounding for each input, product and sum, twice over for silu (slope up to 1.1), and the result's own
        tol = 16 * 2.0 ** -24 * size + 1e-6 + (2.0 ** -8 * y.abs() if dtype == torch.bfloat16 else 0.0)
        assert bool(((got[at:at + lens[s]].double() - y).abs() <= tol).all())
