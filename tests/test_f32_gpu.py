"""The float32 path's products and attention on the matrix cores, alone: at the edges of their tiles, runs and waves,
against float64 arithmetic."""

import math

import numpy as np
import pytest
import torch

from helpers import build_pages
from test_kernels_gpu import attention_ref, close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ops():
    from dryft_amd.csrc import ops as o
    return o


def within_sums(got, x, w, what):
    """Sums of products of random signs in 32 bits. Added one after the other, partial sum j is some sqrt(j) products large and
    is rounded by some 0.4 x 2^-24 of itself, all of them together by 0.3 x 2^-24 |x| |w|: 3.5 of these units are the largest of
    10^5 sums. Operands of 10-bit mantissas are off by 340 units and more at the sizes here, of 16-bit ones by 5."""
    want = x.double() @ w.double().T
    most = 5 * 2.0 ** -24 * x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None, :]
    off = (got.cpu().double() - want).abs()
    assert torch.isfinite(got).all() and (off <= most).all(), f"{what}: {float((off / most).max())} of what sums allow"


@pytest.mark.parametrize("m,n,k,splits", [(1, 1024, 2048, 4), (4, 1000, 3072, 3), (16, 17, 36, 1), (5, 33, 1028, 2),
                                          (3, 2100, 2052, 1), (16, 64, 96, 8), (2, 16, 4, 1)])
def test_gemm_rows_f32_splits(m, n, k, splits):
    torch.manual_seed(m + n + k)
    x, w = torch.randn(m, k), torch.randn(n, k)
    shape = (m, n) if splits == 1 else (splits, m, n)
    out = ops().gemm_rows_f32(x.to(DEV), w.to(DEV), torch.full(shape, float("nan"), device=DEV), splits)
    # the splits' sums are added in 64 bits here, which adds no error
    within_sums(out if splits == 1 else out.double().sum(0), x, w, f"rows {m, n, k, splits}")


@pytest.mark.parametrize("m,inter,k", [(1, 3072, 1024), (16, 9, 36), (4, 1000, 2052), (7, 8, 4)])
def test_gemm_rows_swiglu_f32(m, inter, k):
    torch.manual_seed(m + inter + k)
    x, w = torch.randn(m, k), torch.randn(2 * inter, k) / math.sqrt(k)
    gu = x.double() @ w.double().T
    want = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    out = ops().gemm_rows_swiglu_f32(x.to(DEV), w.to(DEV), torch.full((m, inter), float("nan"), device=DEV))
    close(out, want, torch.float32, what="rows swiglu float32")


@pytest.mark.parametrize("m,n,k", [(17, 64, 32), (129, 65, 96), (33, 130, 1024), (1, 5, 64), (525, 1024, 2048), (64, 127, 160)])
@pytest.mark.parametrize("shape", [-1, 0, 1, 2])
def test_gemm_direct_f32(m, n, k, shape):
    torch.manual_seed(m + n + k)
    x, w = torch.randn(m, k + 4), torch.randn(n, k)                        # rows that are not contiguous
    out = ops().gemm_direct_f32(x.to(DEV)[:, :k], w.to(DEV), torch.full((m, n), float("nan"), device=DEV), shape=shape)
    within_sums(out, x[:, :k], w, f"direct {m, n, k} shape {shape}")


ATTENTION = [  # heads, kv heads, head size, lengths (cached tokens incl. the rows'), rows a sequence, window
    (16, 8, 128, [1, 300, 64, 33], 1, None), (32, 8, 128, [700], 1, None), (4, 2, 16, [17, 9, 200], 1, None),
    (20, 1, 64, [77, 140], 1, None), (6, 3, 48, [100, 129], 1, 33), (4, 2, 256, [130, 31], 1, None),
    (16, 8, 128, [150, 64, 209], 70, None), (6, 3, 48, [129, 90], 64, 40), (8, 2, 32, [31, 13, 6, 1], 31, None),
    (4, 2, 256, [70, 33], 33, 32), (9, 3, 144, [95], 17, None)]


@pytest.mark.parametrize("case", ATTENTION)
@pytest.mark.parametrize("dead", [(), (0,)])
@pytest.mark.parametrize("way", ["rows", "tiles"])
def test_attn_f32(case, dead, way):
    n_heads, n_kv, D, lengths, tq, window = case
    if len(lengths) == 1 and dead:
        pytest.skip("the only sequence cannot sit out")
    torch.manual_seed(D + sum(lengths))
    B, L = len(lengths), max(lengths)
    k, v = torch.randn(B, L, n_kv, D), torch.randn(B, L, n_kv, D)
    q_lens = [min(tq, n) for n in lengths]
    q = torch.randn(B, max(q_lens), n_heads, D)
    q_pos = torch.full((B, max(q_lens)), -1, dtype=torch.long)
    for b, (n, ql) in enumerate(zip(lengths, q_lens)):
        if b not in dead:
            q_pos[b, :ql] = torch.arange(n - ql, n)
    want = attention_ref(q, k, v, lengths, q_pos, D ** -0.5, window)
    k_pages, v_pages, table, slots = build_pages(k, v, lengths, sum((n + 63) // 64 for n in lengths) + 3, B + 2, seed=1, poison=1e4)
    if window:                                   # pages that no row of the step sees any more are gone
        for b, (n, ql) in enumerate(zip(lengths, q_lens)):
            table[slots[b], : max(0, n - ql - window + 1) // 64] = -1
    slots = [-1 if b in dead else s for b, s in enumerate(slots)]
    i32 = lambda values: torch.tensor(np.asarray(values), dtype=torch.int32, device=DEV)
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    packed = torch.cat([q[b, :ql] for b, ql in enumerate(q_lens)]).contiguous().to(DEV)
    out = torch.full_like(packed, float("nan")) if way == "rows" else torch.zeros_like(packed)
    if way == "rows":
        index = dict(row_slot=i32([slots[b] for b, ql in enumerate(q_lens) for _ in range(ql)]),
                     row_pos=i32([int(p) for b, ql in enumerate(q_lens) for p in q_pos[b, :ql]]))
    else:
        tile_cu = np.concatenate([[0], np.cumsum([0 if b in dead else -(-ql // 16) for b, ql in enumerate(q_lens)])])
        index = dict(tiles=(i32(slots), i32(cu), i32(tile_cu), i32([n - ql for n, ql in zip(lengths, q_lens)]), B,
                            int(tile_cu[-1]) + 2))
    ops().attn_f32(packed, k_pages.to(DEV), v_pages.to(DEV), table.to(DEV), out, n_heads, n_kv, D, D ** -0.5, window or 0, **index)
    close(out, torch.cat([want[b, :ql] for b, ql in enumerate(q_lens)]), torch.float32, what=f"attn_f32 {way} {case}")
    for b in dead:
        assert not out[int(cu[b]):int(cu[b + 1])].any()


@pytest.mark.parametrize("D", [32, 128, 256])
@pytest.mark.parametrize("way", ["rows", "tiles"])
def test_attn_f32_scores_without_a_number(D, way):
    """Scores of NaN, +inf and -inf: a row is a number exactly where the softmax over its keys is one (-inf beside other
    scores weighs nothing, also where the first hundreds of keys are of that kind)."""
    n_heads, n_kv = 4, 2
    lengths = [70, 64, 300, 40, 50, 33]
    torch.manual_seed(D)
    B, L = len(lengths), max(lengths)
    k, v, q = torch.randn(B, L, n_kv, D), torch.randn(B, L, n_kv, D), torch.randn(B, L, n_heads, D)
    q[..., 0] = q[..., 0].abs() + 0.1
    endless = lambda sign: torch.tensor([sign * float("inf")] + [0.0] * (D - 1))
    k[0, 40] = float("nan")                       # rows from 40 on
    k[1, 10, 0] = endless(1)                      # of one kv head, rows from 10 on
    k[2, :290] = endless(-1)                      # whole waves without a finite score; from row 290 on there is one
    k[3] = endless(-1)                            # nothing else
    q[4, 7, 1] = float("nan")                     # one query
    q_pos = torch.tensor([[t if t < n else -1 for t in range(L)] for n in lengths])
    want = attention_ref(q, k, v, lengths, q_pos, D ** -0.5)
    k_pages, v_pages, table, slots = build_pages(k, v, lengths, sum((n + 63) // 64 for n in lengths) + 1, B, seed=2, poison=1e4)
    i32 = lambda values: torch.tensor(np.asarray(values), dtype=torch.int32, device=DEV)
    packed = torch.cat([q[b, :n] for b, n in enumerate(lengths)]).contiguous().to(DEV)
    out = torch.zeros_like(packed)
    if way == "rows":
        index = dict(row_slot=i32([s for s, n in zip(slots, lengths) for _ in range(n)]),
                     row_pos=i32([t for n in lengths for t in range(n)]))
    else:
        tiles = [-(-n // 16) for n in lengths]
        index = dict(tiles=(i32(slots), i32(np.concatenate([[0], np.cumsum(lengths)])), i32(np.concatenate([[0], np.cumsum(tiles)])),
                            i32([0] * B), B, sum(tiles)))
    ops().attn_f32(packed, k_pages.to(DEV), v_pages.to(DEV), table.to(DEV), out, n_heads, n_kv, D, D ** -0.5, 0, **index)
    out, want = out.cpu(), torch.cat([want[b, :n] for b, n in enumerate(lengths)])
    assert torch.equal(out.isnan(), want.isnan()) and 0 < int(want.isnan().sum()) < want.numel()
    close(out.nan_to_num(0.0), want.nan_to_num(0.0), torch.float32, what=f"attn_f32 {way}, scores without a number")
