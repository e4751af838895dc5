"""Decoding attention whose queries, key and value come straight from the projection: against 64 bits, and against the kernels it stands
for, the turn and the append to the cache in one launch, attention in another, the gate in a third. The same roundings in the same
places, so pages and outputs differ by the roundings of a differently contracted product at most."""
import math

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


def turned_exactly(x, w, cos, sin, rot, pairs, eps, unit=False):
    """Heads ``x [heads, D]`` normed by ``w`` (None: not), the first ``rot`` features turned, made unit behind that (``unit``), in 64 bits."""
    if w is not None:
        x = x * (x.pow(2).mean(-1, keepdim=True) + eps).rsqrt() * w
    if rot:
        one, two = (x[:, 0:rot:2], x[:, 1:rot:2]) if pairs else (x[:, :rot // 2], x[:, rot // 2:rot])
        first, second = one * cos - two * sin, two * cos + one * sin
        x = torch.cat([torch.stack([first, second], -1).flatten(1) if pairs else torch.cat([first, second], -1), x[:, rot:]], -1)
    return x * (x.pow(2).mean(-1, keepdim=True) + eps).rsqrt() if unit else x


def exact_rows(table, k, v, slots, lens, new, G, scale, window=0, chunk=0, cap=0.0, sink=None, rel=None):
    """Attention of each live sequence's row in 64 bits over pages ``k [pages, G, 64, .]`` and ``v [pages, G, ., 64]``. ``new[i]``: the row's
    queries ``[H, D]``, and its keys and values ``[G, .]`` where they are appended (else None: the pages hold them). Yields the sequence, the
    outputs and, for their error, the sums of ``p |v|`` and the largest product of a feature of q and one of a key that it sees."""
    column = torch.tensor([p // 32 * 32 + 8 * (p % 16 // 4) + 4 * (p % 32 // 16) + p % 4 for p in range(64)])
    for i, (slot, length) in enumerate(zip(slots, lens)):
        if slot < 0:
            continue
        q, own_k, own_v = new[i]
        H, D = q.shape
        held = table[slot, :-(-length // 64)].long()
        keys = k[held][..., :D].permute(0, 2, 1, 3).flatten(0, 1)[:length].double().clone()
        values = v[held][..., column].permute(0, 3, 1, 2).flatten(0, 1)[:length].double().clone()
        if own_k is not None:
            keys[-1], values[-1, :, :own_v.shape[-1]] = own_k, own_v
        pos = length - 1
        lo = pos - pos % chunk if chunk else max(0, length - window) if window else 0
        kh, vh = (t[lo:].repeat_interleave(H // G, 1).permute(1, 0, 2).contiguous() for t in (keys, values))
        sc = (kh * q[:, None]).sum(-1) * scale
        if cap:
            sc = cap * torch.tanh(sc / cap)
        if rel is not None:
            sc = sc + rel.double()[(pos - torch.arange(lo, length)).clamp(max=rel.shape[0] - 1)].T
        p = torch.softmax(sc if sink is None else torch.cat([sc, sink.double()[:, None]], 1), 1)[:, :length - lo, None]
        yield i, (p * vh).sum(1), (p * vh.abs()).sum(1), float((q[:, None] * kh).abs().max())


def room(want, spread, product, scale):
    """How far bfloat16 results may be off: probabilities rounded (2^-9 of each, in sum and total), the result's own rounding, and a feature
    of q or of the new key that lies next to the middle of two bfloat16 numbers rounded the other way (2^-8 of its product in a
    score, which counts twice in the quotient; two of them)."""
    return 2.0 ** -8 * want.abs() + (2.0 ** -8 + 4 * 2.0 ** -8 * product * scale) * spread + 1e-6


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
    x, cpu = src.double().cpu(), lambda t: None if t is None else t.double().cpu()
    new, rounded = {}, lambda t: t.bfloat16().double()
    for i, length in enumerate(LENS):
        tables = (cpu(cos)[length - 1], cpu(sin)[length - 1]) if rot else (None, None)
        heads = [turned_exactly(x[i, a:a + m * D].view(m, D), cpu(w), *tables, rot, what[0] == "pairs", eps, unit)
                 for a, m, w in ((0, H, qw), (H * D, G, kw))]
        new[i] = (rounded(heads[0]), rounded(heads[1]) if write else None, x[i, (H + G) * D:cols].view(G, Dv) if write else None)
    for i, o, spread, product in exact_rows(f["table"].cpu(), k.cpu(), v.cpu(), SLOTS, LENS, new, G, scale, window, chunk, cap,
                                            *(None if t is None else t.cpu() for t in (sink, rel))):
        by = torch.sigmoid(x[i, cols:cols + H * Dv].view(H, P)) if gate is not None else 1.0
        tol = room(o, spread, product, scale) * by + (2.0 ** -8 * (o * by).abs() if gate is not None else 0.0)
        assert bool(((got[i].double().cpu() - o * by).abs() <= tol).all()), i


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
    x = (src.cpu().sum(0).bfloat16() if sums else src.cpu()).double() + (b.double().cpu() if bias else 0.0)
    new, rounded = {}, lambda t: t.bfloat16().double()
    for i, length in enumerate(LENS):
        tables = (cos.double().cpu()[length - 1], sin.double().cpu()[length - 1]) if rot else (None, None)
        q, key = (turned_exactly(x[i, a:a + 2 * m * D].view(2 * m, D), None, *tables, rot, True, eps) for a, m in ((0, H), (2 * H * D, G)))
        new[i] = q, key, rounded(x[i, 2 * (H + G) * D:].view(G, Dv))
    maps = []
    for m in range(2):                              # the maps are attentions of their own on their features of the keys
        km = k[..., m * step_w:m * step_w + D].cpu()
        mine = {i: (rounded(q[m::2]), rounded(key[m::2]) if write else None, val if write else None) for i, (q, key, val) in new.items()}
        maps.append({i: rest for i, *rest in exact_rows(f["table"].cpu(), km, v[:, :, :Dv].cpu(), SLOTS, LENS, mine, G, scale)})
    for i in maps[0]:
        (o1, s1, p1), (o2, s2, p2) = maps[0][i], maps[1][i]
        d = o1 - lam * o2
        by = (d.pow(2).mean(-1, keepdim=True) + eps).rsqrt() * post
        # the difference of the maps' errors, through the norm: its own and that of the root mean square
        tol = (room(o1, s1, p1, scale) + lam * room(o2, s2, p2, scale)) * by
        tol = tol + (d * by).abs() * (tol / post).pow(2).mean(-1, keepdim=True).sqrt() + 2.0 ** -8 * (d * by).abs()
        assert bool(((got[i].double().cpu() - d * by).abs() <= tol).all()), i
