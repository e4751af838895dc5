"""The delta rule and the state-space recurrence sixteen rows at a time, against 64-bit walks row by row: lengths around a
chunk and the ring of chunks, states at the edges of the kernel's two sizes, columns that do not fill a wave, sequences that
sit out, decays that forget at once and that hardly forget, and rows that the general walk takes instead."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENGTHS = (33, 0, 17, 1, 300, 16, 64, 49)       # the second sits out
# float32 sums of up to 128 products and 16 tokens a chunk, a few 2^-24 each; a state that forgets nothing in 300 rows
# carries the roundings of all 19 chunks: 32 x 2^-24 of the outputs' size, the largest of some 10^5 values.
TOL = 64 * 2.0 ** -24


def walk(kind, x, gates, dt_bias, a_log, skip, state, H, G, D, P, eps):
    x, gates = x.double(), gates.double()
    dt = torch.nn.functional.softplus(gates[:, :H] + dt_bias.double())
    decay, beta = torch.exp(-a_log.double().exp() * dt), torch.sigmoid(gates[:, H:])
    q, k = (t.reshape(-1, G, D).repeat_interleave(H // G, 1) for t in (x[:, :G * D], x[:, G * D:2 * G * D]))
    v = x[:, 2 * G * D:].reshape(-1, H, P)
    if kind == "delta":
        unit = lambda t: t / (t.pow(2).sum(-1, keepdim=True) + eps).sqrt()
        q, k = unit(q) * D ** -0.5, unit(k)
    S, out = state.double().clone(), []
    for t in range(x.shape[0]):
        S = S * decay[t][:, None, None]
        u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1)) if kind == "delta" else dt[t][:, None] * v[t]
        S = S + k[t][:, :, None] * u[:, None, :]
        out.append((S * q[t][:, :, None]).sum(1) + (0 if kind == "delta" else skip.double()[:, None] * v[t]))
    return torch.stack(out).flatten(1) if out else x.new_zeros(0, H * P), S


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind,H,G,D,P,rate,pad", [("delta", 4, 2, 128, 128, None, 0), ("delta", 2, 1, 64, 40, -9.0, 8), ("delta", 3, 3, 8, 5, 6.0, 0),
                                                   ("delta", 2, 2, 72, 16, None, 0), ("delta", 2, 1, 64, 32, None, 1), ("state", 4, 2, 128, 64, None, 0),
                                                   ("state", 3, 1, 64, 72, -9.0, 8), ("state", 2, 1, 24, 8, 6.0, 0), ("state", 2, 1, 128, 33, None, 0)])
def test_walk_by_chunks(dtype, kind, H, G, D, P, rate, pad):
    from dryft_amd.csrc import ops
    g = torch.Generator().manual_seed(D + P + H)
    rows, n, eps = sum(LENGTHS), len(LENGTHS), 1e-6
    width = 2 * G * D + H * P
    x = torch.randn(rows, (width + 7) // 8 * 8 + pad, generator=g).to(dtype)
    gates = torch.randn(rows, 2 * H, generator=g)
    dt_bias, skip = torch.randn(H, generator=g), torch.randn(H, generator=g)
    a_log = torch.randn(H, generator=g) if rate is None else torch.full((H,), rate)
    state = torch.randn(n + 2, H, D, P, generator=g)
    slots = [3, -1, 0, 5, 1, 9, 2, 7]
    cu = torch.tensor([0] + torch.tensor(LENGTHS).cumsum(0).tolist(), dtype=torch.int32)
    dev = lambda t: t.to(DEV)
    got_state, out = dev(state.clone()), torch.full((rows, H * P), 7.0, device=DEV)
    facts = (dev(torch.tensor(slots, dtype=torch.int32)), dev(cu), dev(torch.tensor(LENGTHS, dtype=torch.int32)), n, got_state, out)
    seg_cu = torch.tensor([0] + [-(-q // 64) * (s >= 0) for q, s in zip(LENGTHS, slots)]).cumsum(0).to(torch.int32)
    segments = (64, dev(seg_cu), int(seg_cu[-1])) if kind == "delta" else None
    xd = dev(x)
    by_chunks = ops._walks_by_chunks(xd, 0, G * D, D, P, H, n, max(LENGTHS), segments is not None,
                                     ops._DELTA_WALK_US if kind == "delta" else ops._SSM_WALK_US)
    assert by_chunks == (pad != 1)                                    # rows that do not begin at 16 bytes: the general walk
    if kind == "delta":
        ops.delta_steps(xd, 0, G * D, 2 * G * D, dev(gates), 0, H, dev(dt_bias), dev(a_log), *facts, H, G, D, P, D ** -0.5, eps, True,
                        segments=segments, longest=max(LENGTHS))
    else:
        ops.ssm_scan(xd, 2 * G * D, G * D, 0, dev(gates), dev(dt_bias), dev(a_log), dev(skip), *facts, H, P, D, G, True,
                     segments=segments, longest=max(LENGTHS))
    out, got_state = out.double().cpu(), got_state.double().cpu()
    for s, (slot, q) in enumerate(zip(slots, LENGTHS)):
        r = slice(int(cu[s]), int(cu[s]) + q)
        if slot < 0:
            continue
        want, S = walk(kind, x[r, :width], gates[r], dt_bias, a_log, skip, state[slot], H, G, D, P, eps)
        assert float((out[r] - want).abs().max()) <= TOL * float(want.pow(2).mean().sqrt()) * 4, (slot, q)
        assert float((got_state[slot] - S).abs().max()) <= TOL * float(S.pow(2).mean().sqrt()) * 4, (slot, q)
    for slot in set(range(n + 2)) - set(slots):                       # nobody else's state is touched
        assert torch.equal(got_state[slot], state[slot].double())


def drawn(kind, H, G, D, P, lengths, dtype, seed):
    """Inputs of a step of these sequences, each in the slot of its own number."""
    g = torch.Generator().manual_seed(seed)
    rows = sum(lengths)
    return dict(x=torch.randn(rows, (2 * G * D + H * P + 7) // 8 * 8, generator=g).to(dtype), gates=torch.randn(rows, 2 * H, generator=g),
                dt_bias=torch.randn(H, generator=g), a_log=torch.randn(H, generator=g), skip=torch.randn(H, generator=g),
                state=torch.randn(len(lengths), H, D, P, generator=g))


def by_chunks(kind, d, H, G, D, P, lengths, eps):
    """Outputs and states of the step, by chunks."""
    from dryft_amd.csrc import ops
    n, longest = len(lengths), max(lengths)
    dev, ints = (lambda t: t.to(DEV)), (lambda v: torch.tensor(v, dtype=torch.int32, device=DEV))
    x, state, out = dev(d["x"]), dev(d["state"].clone()), torch.full((d["x"].shape[0], H * P), 7.0, device=DEV)
    assert ops._walks_by_chunks(x, 0, G * D, D, P, H, n, longest, False, None)
    facts = (ints(list(range(n))), ints([0] + torch.tensor(lengths).cumsum(0).tolist()), ints(lengths), n, state, out)
    if kind == "delta":
        ops.delta_steps(x, 0, G * D, 2 * G * D, dev(d["gates"]), 0, H, dev(d["dt_bias"]), dev(d["a_log"]), *facts, H, G, D, P, D ** -0.5,
                        eps, True, longest=longest)
    else:
        ops.ssm_scan(x, 2 * G * D, G * D, 0, dev(d["gates"]), dev(d["dt_bias"]), dev(d["a_log"]), dev(d["skip"]), *facts, H, P, D, G, True,
                     longest=longest)
    return out.double().cpu(), state.double().cpu()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,P", [(4, 2, 128, 128), (2, 1, 64, 40), (3, 3, 24, 5)])
def test_unit_vectors_without_an_eps(dtype, H, G, D, P):
    """Lengths that do not fill their last chunk: the zeros that do have no direction, and no say in anything."""
    lengths = (17, 33, 16, 1)
    d = drawn("delta", H, G, D, P, lengths, dtype, D + P)
    out, state = by_chunks("delta", d, H, G, D, P, lengths, 0.0)
    at = 0
    for s, q in enumerate(lengths):
        want, S = walk("delta", d["x"][at:at + q, :2 * G * D + H * P], d["gates"][at:at + q], d["dt_bias"], d["a_log"], d["skip"], d["state"][s],
                       H, G, D, P, 0.0)
        assert float((out[at:at + q] - want).abs().max()) <= TOL * float(want.pow(2).mean().sqrt()) * 4, q
        assert float((state[s] - S).abs().max()) <= TOL * float(S.pow(2).mean().sqrt()) * 4, q
        at += q


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind,H,G,D,P", [("delta", 2, 1, 128, 40), ("delta", 2, 1, 64, 32), ("state", 2, 1, 128, 40), ("state", 2, 2, 24, 32)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_a_bad_row_leaves_the_rows_before_it_alone(kind, H, G, D, P, dtype, bad):
    """One value of one row that is no number (in q, k, v or a gate): what becomes none is what becomes none row by row, in
    outputs and states, and everything else is what it would be."""
    parts = {"q": 1, "k": G * D + 2, "v": 2 * G * D + P - 1, "v2": 2 * G * D + P + 3}
    lengths = (40, 33, 35, 20) + ((18, 50) if bad != bad else ())
    d = drawn(kind, H, G, D, P, lengths, dtype, D + P)
    cu = [0] + torch.tensor(lengths).cumsum(0).tolist()
    for s, (part, row) in enumerate(zip(parts, (21, 16, 18, 9))):
        d["x"][cu[s] + row, parts[part]] = bad
    if bad != bad:
        d["gates"][cu[4] + 5, 0] = bad
        d["gates"][cu[5] + 31, H] = bad                       # of the delta rule alone
    out, state = by_chunks(kind, d, H, G, D, P, lengths, 1e-6)
    lost = 0
    for s, q in enumerate(lengths):
        r = slice(cu[s], cu[s] + q)
        want, S = walk(kind, d["x"][r, :2 * G * D + H * P], d["gates"][r], d["dt_bias"], d["a_log"], d["skip"], d["state"][s], H, G, D, P, 1e-6)
        for got, ref in ((out[r], want), (state[s], S)):
            assert torch.equal(got.isfinite(), ref.isfinite()), (s, (got.isfinite() != ref.isfinite()).nonzero()[:4])
            rest = ref[ref.isfinite()]
            lost += ref.numel() - rest.numel()
            if rest.numel():
                assert float((got[ref.isfinite()] - rest).abs().max()) <= TOL * float(rest.pow(2).mean().sqrt()) * 4, s
    assert lost
