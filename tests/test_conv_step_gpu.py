"""The short convolution of a step of one row a sequence, which moves the tail on itself: equal, bit for bit, to the two
launches it stands for, over the first positions of a sequence, sequences that sit out, and every layout of the weights."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("channels,taps,col", [(1, 2, 0), (255, 4, 3), (256, 4, 8), (520, 3, 0), (257, 16, 1)])
def test_one_row_a_sequence(dtype, channels, taps, col):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(channels + taps)
    slots, positions = [2, -1, 0, 4, 1], [0, 0, 1, taps - 2, 700]
    n = len(slots)
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    u = torch.randn(n, channels + col + 5, generator=g).to(dtype).to(DEV)
    w = torch.randn(channels, taps, generator=g).to(DEV)
    ib, ob = torch.randn(channels, generator=g).to(DEV), torch.randn(channels, generator=g).to(DEV)
    tail = torch.randn(6, taps - 1, channels, generator=g).to(DEV)
    row_slot, row_seq, row_pos, q_len = ints(slots), ints(list(range(n))), ints(positions), ints([int(s >= 0) for s in slots])
    for w_t in (None, w.t().contiguous()):
        for in_bias, out_bias, silu in ((None, None, False), (ib, ob, True)):
            old, new = tail.clone(), tail.clone()
            want, got = (torch.full((n, channels), 9.0, dtype=dtype, device=DEV) for _ in range(2))
            ops.causal_conv(u, col, channels, in_bias, w, out_bias, silu, row_slot, row_seq, row_pos, row_pos, old, want, weight_t=w_t)
            ops.conv_tail(u, col, channels, in_bias, taps, row_slot, ints(list(range(n + 1))), q_len, n, old)
            ops.causal_conv(u, col, channels, in_bias, w, out_bias, silu, row_slot, row_seq, row_pos, row_pos, new, got, weight_t=w_t,
                            moves_tail=True)
            assert torch.equal(got, want) and torch.equal(new, old)
