"""Decoding attention whose queries, key and value come straight from the projection, against the kernels it stands for: the turn and
the append to the cache in one launch, attention in another, the gate in a third. The same roundings in the same places, so pages
and outputs differ by the roundings of a differently contracted product at most."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENS = (1, 33, 64, 7, 65, 300, 96)               # keys with the row's own; the fourth sits out
SLOTS = (2, 0, 7, -1, 5, 1, 3)


def step(G, P, seed, fill=True):
    """Pages of random keys and values with the sequences' tables, and the step's facts."""
    g = torch.Generator().manual_seed(seed)
    n, per = len(LENS), 8
    pages = n * per
    k, v = (torch.randn(pages, G, *shape, generator=g).bfloat16() for shape in ((64, P), (P, 64)))
    order = torch.randperm(pages, generator=g)
    table = torch.full((9, per), -1, dtype=torch.int32)
    for i, (slot, length) in enumerate(zip(SLOTS, LENS)):
        if slot >= 0:
            m = -(-length // 64)
            table[slot, :m] = order[i * per:i * per + m].int()
    dev, ints = (lambda t: t.to(DEV)), (lambda x: torch.tensor(x, dtype=torch.int32, device=DEV))
    facts = dict(table=dev(table), slot=ints(SLOTS), cu=ints(list(range(n + 1))), kv=ints(LENS), pos=ints([x - 1 for x in LENS]))
    return g, n, dev(k), dev(v), facts


def close(a, b):
    """bfloat16 results of the same arithmetic: a query or key feature may round the other way (2^-8 of it)."""
    a, b = a.double().cpu(), b.double().cpu()
    assert bool(torch.isfinite(b).all())
    return float((a - b).abs().max()) <= 2.0 ** -6 * float(b.abs().max()) and float((a - b).pow(2).mean().sqrt()) <= 2.0 ** -10 * float(b.abs().max())


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("write", [True, False])
@pytest.mark.parametrize("form,H,G,D,Dv,P,rot", [
    ("pairs", 8, 2, 128, 128, 128, 128), ("pairs", 5, 1, 64, 64, 64, 24), ("pairs gate", 16, 1, 128, 128, 128, 64), ("pairs", 2, 2, 48, 48, 48, 0),
    ("half", 4, 4, 256, 256, 256, 256), ("half norm", 12, 4, 128, 128, 128, 96), ("half unit", 4, 2, 80, 80, 80, 80),
    ("half norm", 6, 2, 72, 40, 80, 36), ("half sink cap", 9, 3, 64, 64, 64, 64), ("half chunk", 4, 2, 64, 64, 64, 64),
    ("half window rel", 4, 2, 32, 32, 32, 32), ("half gate", 4, 1, 16, 16, 16, 16)])
def test_turn_and_attention(splits, write, form, H, G, D, Dv, P, rot):
    from dryft_amd.csrc import ops
    g, n, k, v, f = step(G, P, D + H)
    dev, what = (lambda t: t.to(DEV)), form.split()
    if P != D or P != Dv:                          # padded pages hold zeros behind a head's features
        k[..., D:], v[:, :, Dv:] = 0, 0
    cols = H * D + G * D + G * Dv
    src = torch.randn(n, cols + (H * Dv if "gate" in what else 0) + 3, generator=g).bfloat16().to(DEV)
    ang = torch.randn(300, max(rot // 2, 1), generator=g)
    cos, sin = (dev(ang.cos()), dev(ang.sin())) if rot else (None, None)
    qw, kw = (dev(torch.randn(D, generator=g)) for _ in range(2)) if "norm" in what else (None, None)
    sink = dev(torch.randn(H, generator=g)) if "sink" in what else None
    rel = dev(torch.randn(20, H, generator=g)) if "rel" in what else None
    cap, chunk, window = 5.0 if "cap" in what else 0.0, 64 if "chunk" in what else 0, 40 if "window" in what else 0
    gate = src[:, cols:cols + H * Dv] if "gate" in what else None
    unit, eps, scale = "unit" in what, 1e-5, D ** -0.5
    parts = lambda: (torch.empty(n, H, splits, P, device=DEV), torch.empty(n, H, splits, 2, device=DEV))
    at = (f["table"], f["slot"], f["cu"], f["kv"], n)
    k1, v1, k2, v2 = k.clone(), v.clone(), k.clone(), v.clone()
    q = torch.zeros(n, H, P, device=DEV, dtype=torch.bfloat16)
    if what[0] == "pairs":
        ops.rope_pairs_kv(src, 0, H * D, (H + G) * D, cos, sin, rot, f["slot"], f["pos"], q, k1, v1, f["table"], write, H, G, D, Dv)
    else:
        ops.norm_rope_half_kv(src, 0, H * D, (H + G) * D, qw, kw, eps, cos, sin, rot, f["slot"], f["pos"], q, k1, v1, f["table"], write,
                              H, G, D, Dv, page_dim=P if P != D or P != Dv else 0, unit_after=unit)
    want, got = torch.full_like(q, 7.0), torch.full_like(q, 7.0)
    ops.attn_split_bf16(q, k1, v1, *at, *parts(), splits, want, H, G, P, scale, window, cap, sink, chunk, rel)
    if gate is not None:
        want = ops.sigmoid_gate(want.view(n, H * P), gate, torch.empty(n, H * P, device=DEV, dtype=torch.bfloat16)).view(n, H, P)
    t = ops.Turned(src, 0, H * D, (H + G) * D, D, Dv, cos, sin, rot, what[0] == "pairs", q_weight=qw, k_weight=kw, eps=eps, unit_after=unit,
                   gate=gate)
    ops.attn_turned_bf16(t, write, k2, v2, *at, *parts(), splits, got, H, G, P, scale, window, cap, sink, chunk, rel)
    assert torch.equal(v1, v2) and close(k2, k1) and int((k1 != k2).sum()) <= 2 + n * G * D // 50
    assert close(got, want) and not got[SLOTS.index(-1)].any()


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("write", [True, False])
@pytest.mark.parametrize("H,G,D,Dv,rot,bias,sums", [(16, 4, 64, 128, 64, True, 0), (8, 1, 64, 128, 32, False, 1), (2, 2, 20, 24, 20, True, 3),
                                                    (6, 2, 128, 256, 0, True, 2)])
def test_turn_and_difference(splits, write, H, G, D, Dv, rot, bias, sums):
    from dryft_amd.csrc import ops
    step_w = -(-D // 8) * 8
    P = -(-max(2 * step_w, Dv) // 16) * 16
    g, n, k, v, f = step(G, P, D + H)
    dev = lambda t: t.to(DEV)
    k[..., D:step_w], k[..., step_w + D:], v[:, :, Dv:] = 0, 0, 0
    cols = 2 * H * D + 2 * G * D + G * Dv
    src, b = dev(torch.randn(sums, n, cols, generator=g) if sums else torch.randn(n, cols, generator=g).bfloat16()), dev(torch.randn(cols, generator=g)) if bias else None
    ang = torch.randn(300, max(rot // 2, 1), generator=g)
    cos, sin = (dev(ang.cos()), dev(ang.sin())) if rot else (None, None)
    lam, post, eps, scale = 0.4, 0.7, 1e-5, D ** -0.5
    parts = lambda: (torch.empty(n, 2 * H, splits, P, device=DEV), torch.empty(n, 2 * H, splits, 2, device=DEV))
    at = (f["table"], f["slot"], f["cu"], f["kv"], n)
    k1, v1, k2, v2 = k.clone(), v.clone(), k.clone(), v.clone()
    q = torch.empty(n, H, 2, P, device=DEV, dtype=torch.bfloat16)
    ops.rope_maps_kv((src, sums) if sums else src, 0, 2 * H * D, 2 * (H + G) * D, b, cos, sin, rot, f["slot"], f["pos"], q, step_w, k1, step_w, v1, f["table"], write,
                     H, G, D, Dv)
    want, got = (torch.full((n, H, Dv), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    ops.attn_split_diff_bf16(q, k1, v1, *at, *parts(), splits, want, H, G, step_w, Dv, scale, 0, lam, post, eps)
    t = ops.Turned(src, 0, 2 * H * D, 2 * (H + G) * D, D, Dv, cos, sin, rot, True, bias=b)
    ops.attn_turned_bf16(t, write, k2, v2, *at, *parts(), splits, got, H, G, P, scale, 0, maps=(step_w, lam, post, eps))
    assert torch.equal(v1, v2) and close(k2, k1) and int((k1 != k2).sum()) <= 2 + n * G * D // 50
    assert close(got, want) and not got[SLOTS.index(-1)].any()
