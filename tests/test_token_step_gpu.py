"""One row a sequence through the delta rule (with its read-out) and the state-space recurrence, against 64-bit walks: the narrowest
and widest states, rows that do not fill the row groups, several heads a group, sequences that sit out or have no row, states left
as they were."""
import pytest
import torch
from test_chunk_walk_gpu import walk

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SLOTS, ROWS = (3, -1, 0, 5, 1, 2), (1, 1, 1, 0, 1, 1)
# float32 sums of up to 256 products, each operand a few 2^-24 off; outputs in bfloat16 round once more.
TOL = 64 * 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("write", [True, False])
@pytest.mark.parametrize("kind,H,G,D,P,rate", [("delta", 4, 2, 128, 128, None), ("delta", 2, 1, 256, 256, None), ("delta", 3, 3, 8, 32, 6.0),
                                               ("delta", 2, 1, 72, 64, -9.0), ("state", 4, 2, 128, 64, None), ("state", 2, 2, 256, 256, -9.0),
                                               ("state", 3, 1, 24, 32, 6.0), ("state", 2, 1, 130, 32, None), ("state", 3, 1, 17, 128, None)])
def test_one_row_a_sequence(dtype, write, kind, H, G, D, P, rate):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(D + P + H)
    n, rows, eps = len(SLOTS), sum(ROWS), 1e-6
    width = 2 * G * D + H * P
    x = torch.randn(rows, width + 3, generator=g).to(dtype)
    gates, gate = torch.randn(rows, 2 * H, generator=g), torch.randn(rows, H * P + 5, generator=g).to(dtype)
    dt_bias, skip, weight = torch.randn(H, generator=g), torch.randn(H, generator=g), torch.randn(H * P, generator=g)
    a_log = torch.randn(H, generator=g) if rate is None else torch.full((H,), rate)
    state = torch.randn(n + 2, H, D, P, generator=g)
    dev, ints = (lambda t: t.to(DEV)), (lambda v: torch.tensor(v, dtype=torch.int32, device=DEV))
    cu = [0] + torch.tensor(ROWS).cumsum(0).tolist()
    got_state = dev(state.clone())
    assert ops.token_step_takes(got_state)
    if kind == "delta":
        out = torch.full((rows, H * P), 7.0, device=DEV, dtype=dtype)
        ops.delta_token(dev(x), 0, G * D, 2 * G * D, dev(gates), 0, H, dev(dt_bias), dev(a_log), ints(SLOTS), ints(cu), ints(ROWS), n,
                        got_state, dev(gate)[:, 5:], dev(weight), eps, out, H, G, D, P, D ** -0.5, eps, write)
    else:
        out = torch.full((rows, H * P), 7.0, device=DEV)
        ops.ssm_scan(dev(x), 2 * G * D, G * D, 0, dev(gates), dev(dt_bias), dev(a_log), dev(skip), ints(SLOTS), ints(cu), ints(ROWS), n,
                     got_state, out, H, P, D, G, write, longest=1)
    out, got_state = out.double().cpu(), got_state.double().cpu()
    for s, (slot, q) in enumerate(zip(SLOTS, ROWS)):
        r = slice(cu[s], cu[s] + q)
        if slot < 0 or not q:
            assert bool((out[r] == (0.0 if kind == "delta" else 7.0)).all())
            continue
        want, S = walk(kind, x[r, :width], gates[r], dt_bias, a_log, skip, state[slot], H, G, D, P, eps)
        tol = TOL * float(want.pow(2).mean().sqrt()) * 4
        if kind == "delta":
            o = want.view(q, H, P)
            by = (o.pow(2).mean(-1, keepdim=True) + eps).rsqrt()
            factor = (by * weight.double().view(H, P) * torch.nn.functional.silu(gate[r, 5:].double()).view(q, H, P)).view(q, H * P)
            want, tol = want * factor, (tol * by.amax() + 1e-5) * factor.abs().amax() / by.amin()
        tol = tol + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 and kind == "delta" else 0.0)
        assert bool(((out[r] - want).abs() <= tol).all()), (slot, float((out[r] - want).abs().max()))
        if write:
            assert float((got_state[slot] - S).abs().max()) <= TOL * float(S.pow(2).mean().sqrt()) * 4, slot
    for slot in range(n + 2):
        if not write or slot not in {s for s, q in zip(SLOTS, ROWS) if q}:
            assert torch.equal(got_state[slot], state[slot].double())
