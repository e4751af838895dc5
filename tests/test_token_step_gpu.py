"""One row a sequence through the delta rule and the matrix memory (with their read-outs) and the state-space recurrence, against 64-bit walks: the narrowest
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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("write", [True, False])
@pytest.mark.parametrize("H,D,P,bias", [(4, 128, 256, 0.0), (2, 256, 64, 9.0), (3, 8, 32, -30.0), (2, 130, 128, 0.0)])
def test_one_row_of_a_matrix_memory(dtype, write, H, D, P, bias):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(D + P + H)
    n, rows, eps, cap, runs = len(SLOTS), sum(ROWS), 1e-6, 15.0, -(-P // 64)
    x = torch.randn(rows, 2 * H * D + 2 * H * P + 3, generator=g).to(dtype)
    gates, weight = torch.randn(rows, 2 * H, generator=g), torch.randn(H * P, generator=g)
    bi, bf = torch.randn(H, generator=g), torch.randn(H, generator=g) + bias       # forget gates: hardly, half, at once
    S0, N0 = torch.randn(n + 2, H, D, P, generator=g), torch.randn(n + 2, H, 1, D, generator=g).repeat(1, 1, runs, 1)
    m0 = torch.randn(n + 2, H, 1, generator=g).repeat(1, 1, runs)
    dev, ints = (lambda t: t.to(DEV)), (lambda v: torch.tensor(v, dtype=torch.int32, device=DEV))
    cu = [0] + torch.tensor(ROWS).cumsum(0).tolist()
    S, N, m, out = dev(S0.clone()), dev(N0.clone()), dev(m0.clone()), torch.full((rows, H * P), 7.0, device=DEV, dtype=dtype)
    ops.mlstm_token(dev(x), 0, H * D, 2 * H * D, 2 * H * D + H * P, dev(gates), dev(bi), dev(bf), cap, ints(SLOTS), ints(cu), ints(ROWS), n,
                    S, N, m, dev(weight), eps, out, H, D, P, D ** -0.5, write)
    out, S, N, m = (t.double().cpu() for t in (out, S, N, m))
    for s, (slot, q) in enumerate(zip(SLOTS, ROWS)):
        r = cu[s]
        if slot < 0 or not q:
            assert slot >= 0 or not out[r].any()
            continue
        xs = x[r].double()
        qv, k = xs[:H * D].view(H, D) * D ** -0.5, xs[H * D:2 * H * D].view(H, D)
        v, gate = (xs[2 * H * D + i * H * P:2 * H * D + (i + 1) * H * P].view(H, P) for i in (0, 1))
        soft = lambda t: cap * torch.tanh(t.double() / cap)
        gi, gf = soft(gates[r, :H].double() + bi.double()), torch.nn.functional.logsigmoid(soft(gates[r, H:].double() + bf.double()))
        mm = torch.maximum(gf + m0[slot, :, 0].double(), gi)
        keep, take = torch.exp(gf + m0[slot, :, 0].double() - mm)[:, None], torch.exp(gi - mm)[:, None]
        want_n = keep * N0[slot, :, 0].double() + take * k
        want_s = keep[:, :, None] * S0[slot].double() + (take * k)[:, :, None] * v[:, None, :]
        o = (want_s * qv[:, :, None]).sum(1) / (torch.maximum((want_n * qv).sum(1).abs(), torch.exp(-mm)) + 1e-6)[:, None]
        by = (o.pow(2).mean(-1, keepdim=True) + eps).rsqrt() * weight.double().view(H, P) * torch.sigmoid(gate)
        # the read-out's sums as in TOL, of each head's own size after its norm (the normaliser's error cancels in the norm)
        tol = TOL * 4 * by.abs().amax() / (o.pow(2).mean(-1) + eps).rsqrt().amin() * (o.pow(2).mean(-1) + eps).rsqrt().amax() + 1e-5
        tol = tol + ((o * by).abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0.0)
        assert bool(((out[r].view(H, P) - o * by).abs() <= tol).all()), (slot, float((out[r].view(H, P) - o * by).abs().max()))
        if write:
            assert float((S[slot] - want_s).abs().max()) <= TOL * 4 * float(want_s.pow(2).mean().sqrt()) + TOL
            assert float((N[slot] - want_n[:, None]).abs().max()) <= TOL * 4 and float((m[slot] - mm[:, None]).abs().max()) <= TOL * 4
    for slot in range(n + 2):
        if not write or slot not in {s for s, q in zip(SLOTS, ROWS) if q}:
            assert all(torch.equal(a[slot], b[slot].double()) for a, b in ((S, S0), (N, N0), (m, m0)))


@pytest.mark.parametrize("write", [True, False])
@pytest.mark.parametrize("rows,size,taps", [(1, 128, 4), (5, 32, 1), (16, 96, 5), (17, 256, 4), (33, 128, 16), (17, 160, 2)])
def test_one_row_of_a_gated_linear_recurrence(write, rows, size, taps):
    """Against the formulas in 64 bits; the convolution is rounded to bfloat16 where the gates multiply it, on both sides."""
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(rows + size)
    blocks, scale = 3, 8.0
    W = blocks * size
    proj = torch.randn(rows, 2 * W + 5, generator=g).bfloat16()
    xb, yb, cb, ab, ib, lam = (torch.randn(W, generator=g) for _ in range(6))
    conv, tail, S = torch.randn(W, taps, generator=g), torch.randn(rows + 1, max(taps - 1, 1), W, generator=g), torch.randn(rows + 1, W, generator=g)
    wa, wi = ((torch.randn(blocks, size, size, generator=g) * size ** -0.5).bfloat16() for _ in range(2))
    slots = torch.randperm(rows + 1, generator=g)[:rows]
    slots[rows // 2] = -1 if rows > 1 else slots[0]
    dev = lambda t: t.to(DEV)
    got_s, got_t, out = dev(S.clone()), dev(tail.clone()), torch.full((rows, W), 7.0, device=DEV, dtype=torch.bfloat16)
    wad, wid, vectors = dev(wa), dev(wi), [dev(v) for v in (ab, ib, lam, yb)]
    assert ops.rglru_token_takes(dev(proj), got_s, wad, wid, vectors, blocks)
    ops.rglru_token(dev(proj), W, 0, dev(xb), vectors[3], dev(conv), dev(cb), taps, wad, vectors[0], wid, vectors[1], vectors[2], scale,
                    dev(slots.int()), got_s, got_t if taps > 1 else None, out, W, blocks, write)
    out, got_s, got_t = (t.double().cpu() for t in (out, got_s, got_t))
    live = slots >= 0
    assert not out[~live].any()
    rs, at, p = live.nonzero()[:, 0], slots[live], proj.double()
    window = torch.cat([tail.double()[at][:, :taps - 1], (p[rs, W:2 * W] + xb.double())[:, None]], 1)
    u = cb.double() + (window * conv.double().t()).sum(1)
    ub = u.float().bfloat16().double().view(-1, blocks, size)
    gate = lambda w, b: torch.sigmoid((ub.transpose(0, 1) @ w.double().transpose(1, 2).contiguous()).transpose(0, 1).reshape(-1, W) + b.double())
    log_a = -scale * torch.nn.functional.softplus(lam.double()) * gate(wa, ab)
    want_s = log_a.exp() * S.double()[at] + (-torch.expm1(2 * log_a)).sqrt() * gate(wi, ib) * u
    want = want_s * torch.nn.functional.gelu(p[rs, :W] + yb.double(), approximate="tanh")
    # sums of up to 256 float products; an input of the gates whose float sum lies next to a boundary of bfloat16 may round the other way
    # (2^-8 of it, times a weight of size^-1/2, through a slope of scale * softplus * 1/4 at most)
    tol = 2.0 ** -8 * 4 * size ** -0.5 * scale * float(torch.nn.functional.softplus(lam).max()) / 4 * float(want_s.abs().max())
    assert float((out[live] - want).abs().max()) <= tol + 2.0 ** -8 * float(want.abs().max())
    if write:
        assert float((got_s[at] - want_s).abs().max()) <= tol and float((got_s[at] - want_s).pow(2).mean().sqrt()) <= 1e-3
        if taps > 1:
            assert float((got_t[at] - window[:, 1:]).abs().max()) <= 2.0 ** -20
    untouched = [s for s in range(rows + 1) if not write or s not in at.tolist()]
    assert torch.equal(got_s[untouched], S.double()[untouched]) and torch.equal(got_t[untouched], tail.double()[untouched])
