"""Float32 decoding attention whose keys go over several workgroups: against 64 bits, against one workgroup a row, where scores are no
numbers, and with the counters of one launch used again by the next."""
import pytest
import torch
from test_attn_turned_gpu import exact_rows, turned_exactly

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LENS = (1, 33, 700, 96, 129, 260)
SLOTS = (2, 0, 7, -1, 5, 1)


def pages_of(G, D, seed):
    g = torch.Generator().manual_seed(seed)
    per = -(-max(LENS) // 64)
    k, v = torch.randn(len(LENS) * per, G, 64, D, generator=g), torch.randn(len(LENS) * per, G, D, 64, generator=g)
    order, table = torch.randperm(len(LENS) * per, generator=g), torch.full((9, per), -1, dtype=torch.int32)
    for i, (slot, n) in enumerate(zip(SLOTS, LENS)):
        if slot >= 0:
            table[slot, :-(-n // 64)] = order[i * per:i * per + -(-n // 64)].int()
    return g, k, v, table


@pytest.mark.parametrize("splits", [2, 5, 32])
@pytest.mark.parametrize("window", [0, 40])
@pytest.mark.parametrize("H,G,D", [(16, 8, 128), (4, 1, 64), (20, 1, 32), (4, 4, 256), (6, 2, 144), (2, 1, 16)])
def test_keys_over_workgroups(H, G, D, window, splits):
    from dryft_amd.csrc import ops
    g, k, v, table = pages_of(G, D, H + D)
    n = len(LENS)
    q = torch.randn(n, H, D, generator=g).to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    kd, vd, td = k.to(DEV), v.to(DEV), table.to(DEV)
    facts = dict(row_slot=i32(SLOTS), row_pos=i32([x - 1 for x in LENS]))
    one, counters = torch.full_like(q, 7.0), torch.zeros(ops.split_arrivals(n, H, G), dtype=torch.int32, device=DEV)
    ops.attn_f32(q, kd, vd, td, one, H, G, D, D ** -0.5, window, **facts)
    for _ in range(3):
        got = torch.full_like(q, 7.0)
        ops.attn_f32(q, kd, vd, td, got, H, G, D, D ** -0.5, window, splits=splits, arrivals=counters, **facts)
        # sums of the same products in another order: 700 keys, a few 2^-24 each, of values near 1
        assert float((got - one).abs().max()) <= 32 * 2.0 ** -24 and not counters.any()
    assert not got[SLOTS.index(-1)].any()
    pos_of = torch.empty(64, dtype=torch.long)                       # the column of a page of values in which a position lies
    for p in range(64):
        b, r = p // 32 * 32, p % 32
        pos_of[p] = b + 8 * (r % 16 // 4) + 4 * (r // 16) + r % 4
    for i, (slot, length) in enumerate(zip(SLOTS, LENS)):
        if slot < 0:
            continue
        held = table[slot, :-(-length // 64)].long()
        keys = k[held].permute(0, 2, 1, 3).reshape(-1, G, D)[:length].double()
        values = v[held][..., pos_of].permute(0, 3, 1, 2).reshape(-1, G, D)[:length].double()
        lo = max(0, length - window) if window else 0
        for h in range(H):
            s = (keys[lo:, h // (H // G)] @ q[i, h].double().cpu()) * D ** -0.5
            want = torch.softmax(s, 0) @ values[lo:, h // (H // G)]
            assert float((got[i, h].double().cpu() - want).abs().max()) <= 64 * 2.0 ** -24


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_scores_without_a_number(bad):
    """A key that is no number shows in the row whichever workgroup meets it, as with one workgroup a row."""
    from dryft_amd.csrc import ops
    H, G, D = 4, 2, 64
    g, k, v, table = pages_of(G, D, 3)
    q = torch.rand(len(LENS), H, D, generator=g).to(DEV) + 0.1
    k[table[7, 4].long(), :, 9] = bad
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    facts = dict(row_slot=i32(SLOTS), row_pos=i32([x - 1 for x in LENS]))
    one, got = torch.full_like(q, 7.0), torch.full_like(q, 7.0)
    at = (q, k.to(DEV), v.to(DEV), table.to(DEV))
    ops.attn_f32(*at, one, H, G, D, D ** -0.5, 0, **facts)
    ops.attn_f32(*at, got, H, G, D, D ** -0.5, 0, splits=8, **facts)
    assert torch.equal(got.isfinite(), one.isfinite()) and got[3].eq(0).all() and got[0].isfinite().all()
    assert float((got.nan_to_num(0.0, 0.0, 0.0) - one.nan_to_num(0.0, 0.0, 0.0)).abs().max()) <= 32 * 2.0 ** -24


def test_where_keys_are_split():
    from dryft_amd.parts.attention import float32_splits
    assert float32_splits(1, 16, 8, 4096) == 32 and float32_splits(4, 16, 8, 512) == 8 and float32_splits(8, 16, 8, 4096) == 4
    assert float32_splits(4, 16, 8, 40) == 1 and float32_splits(16, 16, 8, 4096) == 1 and float32_splits(1, 40, 1, 4096) == 32


@pytest.mark.parametrize("write", [True, False])
@pytest.mark.parametrize("splits", [1, 4, 32])
@pytest.mark.parametrize("H,G,D,normed,window", [(16, 8, 128, True, 0), (16, 1, 64, False, 0), (6, 3, 96, True, 40), (4, 4, 32, True, 0), (20, 4, 128, False, 33)])
def test_turn_and_attention_in_one(H, G, D, normed, window, splits, write):
    """Against 64 bits, and against the launch of its own for norm, turn and append and then one workgroup a row: float32 throughout."""
    from dryft_amd.csrc import ops
    if D == 128:
        splits = max(splits, 2)                    # unsplit, heads of 128 keep the two launches
    g, k, v, table = pages_of(G, D, H + D)
    n = len(LENS)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    qkv = torch.randn(n, (H + 2 * G) * D + 4, generator=g).to(DEV)
    ang = torch.randn(max(LENS), D // 2, generator=g)
    cos, sin, td = ang.cos().to(DEV), ang.sin().to(DEV), table.to(DEV)
    qw, kw = (torch.randn(D, generator=g).to(DEV) for _ in range(2)) if normed else (None, None)
    facts = dict(row_slot=i32(SLOTS), row_pos=i32([x - 1 for x in LENS]))
    k1, v1, k2, v2 = (t.to(DEV).clone() for t in (k, v, k, v))
    q, want, got = (torch.full((n, H, D), 7.0, device=DEV) for _ in range(3))
    assert ops.attn_f32_fused_takes(qkv, qw, kw, cos, sin, D, k2, v2, H, G, D, splits)
    ops.qk_norm_rope_kv(qkv, qw, kw, 1e-6, cos, sin, D, facts["row_slot"], facts["row_pos"], q, k1, v1, td, write, H, G, D)
    ops.attn_f32(q, k1, v1, td, want, H, G, D, D ** -0.5, window, **facts)
    ops.attn_f32_fused(qkv, qw, kw, 1e-6, cos, sin, write, k2, v2, td, facts["row_slot"], facts["row_pos"], got, H, G, D, D ** -0.5, window,
                       splits=splits)
    # keys: products of two values of a few units, rounded once or twice more; scores of 128 of those, softmax weights of at most 1
    assert torch.equal(v1, v2) and float((k1 - k2).abs().max()) <= 16 * 2.0 ** -24 * float(k1.abs().max())
    assert int((k2 != k.to(DEV)).any(-1).sum()) == (sum(s >= 0 for s in SLOTS) * G if write else 0)
    assert float((got - want).abs().max()) <= 256 * 2.0 ** -24 * float(want.abs().max()) and not got[SLOTS.index(-1)].any()
    x, new, cpu = qkv.double().cpu(), {}, lambda t: None if t is None else t.double().cpu()
    for i, length in enumerate(LENS):
        at = (cpu(cos)[length - 1], cpu(sin)[length - 1], D, False, 1e-6)
        q, key = (turned_exactly(x[i, a:a + m * D].view(m, D), cpu(w), *at) for a, m, w in ((0, H, qw), (H * D, G, kw)))
        new[i] = (q, key, x[i, (H + G) * D:(H + 2 * G) * D].view(G, D)) if write else (q, None, None)
    for i, o, spread, product in exact_rows(table, k, v, SLOTS, LENS, new, G, D ** -0.5, window):
        # a score is a sum of D products of values with some 16 roundings of 2^-24 each behind them (sum of squares, norm, turn), as large as the
        # largest times D^1/2 where they fall either way, times the scale D^-1/2; that counts twice in the quotient, and its sums add theirs
        tol = 2.0 ** -24 * (4 * 16 * product + 64) * spread
        assert bool(((got[i].double().cpu() - o).abs() <= tol).all()), (i, float(((got[i].double().cpu() - o).abs() / tol).max()))
