"""``y = x @ W.T`` for weights in checkpoint layout ``[out, in]`` (no bias).

The reference hands every projection to a vendor library (F.linear,
engine/dryft_qwen3/model.py:153, 179-180, 237, 258-261). Here:

* float32: this library's own kernels, so the 32-bit path has no reduced-precision matrix
  mode anywhere: up to 4 rows the kernel of whole lines (below, on the 32-bit instruction); else the matrix cores' full-precision instruction (``v_mfma_f32_16x16x4_f32``),
  with K split over a workgroup's waves (or plain multiply-adds, ``streams_f32``) for at most 16 rows, operands straight
  into LDS in blocks chosen by the number of workgroups for more (``K`` a multiple of 32; else blocks of
  128 x 128 through registers), and a plain tiled kernel for sizes those do not take;
* bfloat16, at most 16 rows (decoding at small batch): this library's kernel whose loads bring whole cache lines that are
  matrix-core operands as they are, with K split over a workgroup's waves (``lines_pay``), or its weight-streaming
  matrix-core kernel, which stages whole cache lines through LDS and can leave its result
  as float32 partial sums over K for the consumer to add;
* the gated units of feed-forwards at most 16 rows likewise (``ops.gemm_few_glu_ok``);
* bfloat16, at most 96 rows, the fused gate/up product with its activation: this library's kernel that brings
  its operands straight into LDS (``panel_swiglu_ok``; K a multiple of 128, else the two kernels below);
* bfloat16, 17 to 128 rows, where the consumer adds partial sums (q/k/v of decoding steps and short prompts, the projections
  back to the hidden width) or the result is wanted in float32 (the output head), K a multiple of 64: this library's kernel
  that brings its operands straight into LDS, K split over workgroups (``mid_plan``);
* bfloat16, 17 to 64 rows, such products of other K, and sizes the vendor library does not take: this library's
  shared-activation kernel;
* bfloat16, 129 to 256 rows (short prompts, decoding at large batch; large matrices from 65) where the consumer adds partial sums
  and K is a multiple of 64: this library's kernel whose waves each own rows of x, operands straight into LDS (``tall_plan``);
  the fused gate/up product of 97 to 256 rows goes to its other form (``tall_swiglu_ok``), of more rows to this library's
  kernel of 256 rows a workgroup where its rounds of workgroups are nearly full (``many_glu_ok``);
* bfloat16, more than 16 rows, float32 results of at most 64 outputs (gates, routers, low-rank projections): this
  library's kernel that reads the rows once and splits K over the waves of a workgroup;
* bfloat16, otherwise (prompts, decoding at large batch): the vendor library through
  ``torch.mm``, as in the reference; float32 results of many rows and output sizes the
  library does not take are this library's block kernel (128 x 128 or 256 x 256 outputs
  per workgroup, about 0.6 of the library's speed), and what no matrix-core kernel takes goes
  to the plain kernel.
"""

from __future__ import annotations

import contextlib
import functools
import os
import tempfile

import torch

from ..csrc import ops
from .base import Partials

STREAM_ROWS = 16                # the most rows the line-staging kernel takes; up to here it beats the vendor library
WIDE_ROWS = 64                  # the most rows the shared-activation kernel takes
_SMALL_MID_BYTES = 48 << 20     # the largest matrix for which workgroups of 64 outputs come into question
_STREAM_BLOCKS_PER_WAVE = 5     # measured on the projection shapes of 4B to 32B models inside captured graphs:
_STREAM_WORKGROUPS = 1536       # short walks over K, as long as the launch stays under about six workgroups a unit
_COMPUTE_UNITS = 256            # of the MI355X


@functools.lru_cache(maxsize=1024)           # asked at every product of a step
def stream_plan(n: int, k: int, may_split: bool) -> tuple[int, int, int]:
    """(splits of K across workgroups, blocks per group, groups in flight) for the line-staging kernel.

    Splitting pays only where the consumer adds the partial sums up on its way (a pass of their own
    costs more than the split gains).
    """
    tiles = (n + 15) // 16
    k_blocks = (k + 63) // 64
    want = (k_blocks + 4 * _STREAM_BLOCKS_PER_WAVE - 1) // (4 * _STREAM_BLOCKS_PER_WAVE)
    splits = max(1, min(want, _STREAM_WORKGROUPS // tiles, k_blocks // 8, 16)) if may_split else 1
    return (splits, 1, 2) if splits > 1 else (1, 2, 2)


def rows_f32_splits(n: int, k: int) -> int:
    """Splits of K across workgroups for at most 16 rows of float32 values (16 outputs a workgroup): as many as give every
    compute unit a workgroup, each at least 512 values of K."""
    return max(1, min(_COMPUTE_UNITS // ((n + 15) // 16), k // 512, 16))


def streams_f32(m: int, n: int, k: int) -> bool:
    """Does a product of at most 16 rows of float32 values that is not the kernel's of whole lines (up to four rows: ``lines_pay_f32``)
    go to the plain multiply-adds that read whole lines, or to the matrix cores with K split over a workgroup's waves? The first is bound by its arithmetic, the rows of x, and by K walked
    chunk by chunk; the second by its trips to memory (three of them from K = 2,560 on) and by reading the rows of x again in
    every workgroup. In a captured chain on rotating cold weights, us, first against second: 6,144 x 1,024 at 1 / 4 / 8 / 16
    rows 7.2 / 9.3 / 11.8 / 17.3 against 9.0 / 9.8 / 10.5 / 12.3; 4,096 x 1,024 5.8 / 8.0 / 10.3 / 15.7 against 6.4 / 6.6 / 6.9 /
    7.7; 151,936 x 1,024 105 / 120 / 183 / 352 against 136 / 139 / 155 / 182; 19,456 x 2,560 37 / 43 / 52 / 96 against 54 / 58 /
    64 / 78; 2,560 x 9,728 29 / 41 / 48 / 70 against 35 / 37 / 42 / 50."""
    return m <= 2 or (m <= 8 and n >= 6144 and k >= 2560)


def swiglu_f32_ok(h: torch.Tensor, w_gate_up: torch.Tensor) -> bool:
    """Does the float32 gate/up product run with its activation in one kernel? Up to four rows always; beyond, the matrix cores'
    form only, so up to eight rows not from K = 2,560 on: 19,456 x 2,560 at 4 rows 56 us against 43 and 3 for the activation; 6,144 x 1,024 9.9 against
    9.3 and 3."""
    return ops.lines_ok(h, w_gate_up) or \
        (h.shape[0] <= STREAM_ROWS and ops.rows_f32_ok(h, w_gate_up) and not (h.shape[0] <= 8 and h.shape[1] >= 2560))


@functools.lru_cache(maxsize=1024)
def lines_pay(m: int, n: int, k: int, added: bool = False) -> bool:
    """Does a product of at most 16 rows go to the kernel that loads matrix-core operands as whole lines (figures beside it), or
    to the line-staging one? (``added``: where that may leave partial sums that the consumer adds.) Every workgroup of the
    first reads the rows of x again and walks all of K, a workgroup of the second more weight rows for them. In a captured
    chain on rotating cold weights (4 GB), us, first against second:

    * up to eight rows the first is ahead, but for heads of little depth (151,936 x 512 at 8 rows 31.2 / 31.0) and, at five and
      more, large deep matrices whose workgroups of 20 weight rows leave their last round half empty (6,144 x 14,336 with the
      norm behind 43.9 / 40.5);
    * few outputs of a deep K are a long walk for few workgroups, which partial sums cut: with the norm behind, 256 x 14,336 at 8
      rows 10.8 / 8.4, 1,280 x 14,336 16.2 / 14.2 (1,536 16.3 / 15.6: the line), 256 x 25,600 at 4 rows 11.9 / 9.7;
    * at 9 to 16 rows the first is ahead on matrices that leave either a launch's ends (at 16, 2,048 x 2,048 4.6 / 6.1, 3,072 x 2,048
      5.1 / 6.4, 4,096 x 1,024 4.3 / 5.0; beyond 8,192 outputs it has too many workgroups for that, 10,240 x 512 at 9 6.0 / 4.6) and
      on large ones of much depth whose workgroups of 20 weight rows fill their rounds (at 16, 5,120 x 8,192 18.3 / 24.4, 10,240
      x 5,120 23.1 / 25.8, 14,336 x 8,192 45.8 / 52.1, 28,672 x 8,192 88 / 91; half-filled rounds 6,144 x 8,192 with the norm behind
      32.0 / 28.3, 12,288 x 4,096 26.0 / 20.2; less depth 28,672 x 2,048 at 9 rows 31.5 / 22.4, 65,536 x 2,048 65 / 49, 151,936 x 2,560
      176 / 142 and at 16 194 / 167), behind between them (8,192 x 2,048 9.9 / 8.6)."""
    if added and k > 8192 and n <= 1280 and (m > 4 or (k > 16384 and n <= 768)):
        return False
    if m <= 4:
        return True
    if k <= 1024 and n > 32768:
        return False
    if n * k < _LINES_LARGE:
        return m <= 8 or (n * k <= _LINES_SMALL and n <= 8192)
    workgroups = -(-n // 20)
    filled = workgroups / (-(-workgroups // _COMPUTE_UNITS) * _COMPUTE_UNITS)
    if m <= 8:
        return filled >= 0.65 or k <= 8192
    return filled >= 0.85 and k >= (5120 if n <= 16384 else 8192)


_LINES_SMALL, _LINES_LARGE = 8 << 20, 40 << 20


def lines_pay_f32(m: int, n: int, k: int) -> bool:
    """The same for at most four rows of float32 values, against the plain multiply-adds: behind only at one and two rows of many
    outputs and little depth, where a workgroup is mostly its ends (us, 151,936 outputs: K = 256 at one row 36.4 / 28.4, at two
    36.6 / 33.3, K = 512 55 / 50 and 55 / 52; 768 74 / 75; 28,672 of 512 13.0 / 12.6: the line)."""
    return k > 512 or m > 2 or n <= 28672 * m


def wide_plan(n: int, k: int, may_split: bool) -> tuple[int, int, int]:
    """(splits of K across workgroups, blocks per group, groups in flight) for the shared-activation kernel.

    Its workgroups are bound by their own compute unit (LDS and barriers), not by memory, so where the
    consumer adds partial sums the split of K is chosen to give every compute unit one workgroup; measured
    on the o and down shapes of 4B, 8B and 32B models at 24 and 64 rows.
    """
    tiles = (n + 63) // 64
    k_blocks = (k + 63) // 64
    splits = max(1, min(_COMPUTE_UNITS // tiles, k_blocks // 4, 16)) if may_split else 1
    return (splits, 1, 3) if splits > 1 else (1, 2, 1)


def tall_plan(m: int, n: int, k: int) -> tuple[int, int]:
    return _tall_plan(128 if m <= 128 else 256, n, k)


@functools.lru_cache(maxsize=None)
def _tall_plan(loaded: int, n: int, k: int) -> tuple[int, int]:
    """(tiles of 16 outputs a workgroup, splits of K across workgroups) for the product of 65 to 256 rows whose waves
    each own rows of x: the pair with the lowest modelled time. The model, fitted (to 4 % in the mean) to in-graph
    times on rotating cold weights of the q/k/v, o and down shapes of Qwen3-0.6B, 4B, 8B and 14B at 128 and 256 rows,
    every tile count with four to five split counts each, in us (the rows counted as the 128 or 256 the kernel loads):
    3.2 + rounds * (11.1 * MB of x a workgroup takes in + 22.5 * MB of W it takes in) + 0.23 * MB of partial sums
    + 0.074 * MB of W, rounds being how often the workgroups fill the 256 compute units. (A workgroup takes in all
    rows of x, 128 or 256 of them, over its run of K: that is what the time goes to, and why a split pays also where
    the outputs alone would fill the chip.) Its choice is within 5 % of the best measured pair for each of those
    shapes. The choice itself counts 0.42 us a MB of partial sums: the kernel that adds them up on its way in takes
    0.19 us a MB more to read them (the norm after o and down at 256 rows: 6.9 us with eight parts, 21 MB; the
    cache writer after q/k/v 12.0 us with four parts, 7.8 without). Against the kernel it replaces here (64 outputs a workgroup, every wave reading all rows of x from LDS),
    at 256 rows: Qwen3-4B's down 22.5 against 26.8, Qwen3-8B's 34.7 against 59.8, Qwen3-14B's 55.3 against 96.2."""
    groups = k // ops.TALL_GROUP
    best, best_cost = (4, 1), float("inf")
    for tiles in (4, 5, 6, 7, 8):
        blocks = -(-n // (16 * tiles))
        seen = set()
        for want in range(1, min(groups, 32) + 1):
            splits = ops.gemm_mid_splits(k, want)
            if splits in seen:
                continue
            seen.add(splits)
            per = -(-groups // splits)
            rounds = -(-(blocks * splits) // _COMPUTE_UNITS)
            cost = 3.2 + rounds * (11.1 * loaded + 22.5 * 16 * tiles) * per * 128e-6 + 0.42e-6 * splits * loaded * n * 4 + \
                0.074e-6 * n * k * 2
            if cost < best_cost:
                best, best_cost = (tiles, splits), cost
    return best


def small_mid_plan(n: int, k: int) -> int:
    """Splits of K that give every compute unit one workgroup of 64 outputs: what ``mid_plan`` weighs wider workgroups
    against. 1 beyond 48 MiB, where those are always ahead."""
    if n * k * 2 > _SMALL_MID_BYTES:
        return 1
    blocks = (n + 63) // 64
    return ops.gemm_mid_splits(k, max(1, min(16, _COMPUTE_UNITS // blocks)))


def mid_pays(m: int, n: int, k: int, may_split: bool) -> bool:
    """Does a product of 17 to 128 rows go to the kernel of ``mid_plan``, or beyond 64 rows to the one whose waves own rows of x? To
    the first, but for split products of large matrices (5,120 x 25,600, 250 MiB, at 77 / 96 / 128 rows 59 / 69 / 80 us against
    54 / 58 / 63; 5,120 x 17,408, 170 MiB, 36 / 38 / 42 against 38 / 40 / 43) and beyond 96 rows of small ones, whose partial sums
    weigh more than they (steps of 128 sequences through Qwen3-0.6B, 4 to 8 MiB, 2,295 against 2,284 us; Qwen3-4B's, 12 layers,
    20 MiB on, 1,707 against 1,812). Whole float32 results of any size: 200 of 65 to 4,096 outputs (routers) take 0.62 of the time that
    ``gemm_wide`` and ``gemm_block`` took, 0.86 at most, 55 heads of up to 160,000 outputs 0.74. Split products with the norm behind, 800
    sizes: 0.97 on average; 19, of less than 8 MiB but for one, are 3 to 8 % slower than before."""
    size = n * k * 2
    return m <= WIDE_ROWS or not may_split or (size <= 192 << 20 and (m <= 96 or size >= 16 << 20))


def mid_plan(m: int, n: int, k: int, may_split: bool) -> tuple[int, int]:
    return _mid_plan(-(-m // 16) if m <= 96 else 8, n, k, may_split)


@functools.lru_cache(maxsize=1024)
def _mid_plan(tiles: int, n: int, k: int, may_split: bool) -> tuple[int, int]:
    """(waves of 16 outputs a workgroup, splits of K across workgroups) for the kernel that brings its operands straight into
    LDS, with ``tiles`` of 16 rows of x: the pair with the lowest modelled time, in us: 3 + rounds * (30 * MB of W a workgroup
    takes in + 10 * MB of x it takes in) + 0.6 * MB of partial sums, rounds being how often the workgroups fill the compute
    units. Fitted to times in a captured chain on rotating cold weights of 19 sizes (1,024 x 1,024 to 5,120 x 25,600) at
    17 to 128 rows, where partial sums count 0.3; its choice is there within 3 % of the best pair on average (worst 12 %), and
    14 % ahead of what served these sizes before. The kernel that adds them up on its way in counts for the rest: steps of 64
    / 96 sequences through Qwen3-0.6B 1,587 / 2,032 us with 0.3, 1,558 / 1,982 with 0.6, 1,555 / 1,972 with 0.8, of 128 through
    Qwen3-4B (12 layers) 1,732, 1,707 and 1,716. Four waves leave no unit without a workgroup (2,048 x 2,048 at 96 rows, 8 splits 5.9 us, the modelled 4 6.7;
    4,096 x 12,288, 8 waves 27.2, 4 with 4 splits 31.0) but for outputs so few that sixteen splits are needed for that: 1,024 x 3,072 at
    64 rows, 16 / 12 splits 4.53 / 4.55, 5 waves 5.09; steps of 48 / 64 / 96 sequences through Qwen3-0.6B 3 % less than with wider
    workgroups there. Against ``gemm_wide`` at 17 to 32 rows, 64 rows a workgroup and three stages at 33 to
    64, and ``gemm_tall`` beyond, us: 6,144 x 2,560 at 17 / 32 / 64 / 96 rows 8.2 / 8.7 / 10.0 / 11.5 (10.2 / 10.9 / 11.7 / 13.2),
    2,560 x 9,728 10.5 / 11.1 / 12.8 / 14.7 (13.1 / 12.9 / 14.5 / 15.7), 4,096 x 1,024 4.0 / 4.2 / 5.0 / 5.7 (5.3 / 5.8 / 5.0 / 7.0),
    10,240 x 5,120 19.7 / 21.0 / 23.8 / 26.2 (36.6 / 35.5 / 42.2 / 27.5)."""
    groups = k // ops.MID_GROUP
    best, best_cost = (4, 1), float("inf")
    for waves in ops.MID_WAVES:
        blocks = -(-n // (16 * waves))
        fills = waves == 4 and blocks * 16 > _COMPUTE_UNITS      # one workgroup for each unit and no fewer: see above
        wants = (1,) if not may_split else (small_mid_plan(n, k),) if fills else range(1, min(groups, 16) + 1)
        for splits in {ops.gemm_mid_splits(k, want) for want in wants}:
            rounds = -(-(blocks * splits) // _COMPUTE_UNITS)
            if splits > 1 and rounds > 1:
                continue
            cost = rounds * 16 * (30 * waves + 10 * tiles) * -(-groups // splits) * 128e-6 + 0.6e-6 * splits * 16 * tiles * n * 4
            if cost < best_cost:
                best, best_cost = (waves, splits), cost
    return best


def few_rows_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Can the few-row kernels read these operands? (16-byte pieces of rows.)"""
    return x.shape[1] % 8 == 0 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0


def panel_swiglu_ok(x: torch.Tensor, w_gate_up: torch.Tensor) -> bool:
    """Does the fused gate/up product with its activation go to the kernel that brings its operands straight into
    LDS? K a multiple of its group, up to 64 rows, and up to 96 where the matrix is at most 384 MiB. In-graph times on
    rotating cold weights, us, against the line-staging kernel (up to 16 rows) or the vendor library plus the activation
    kernel (more), Qwen3-4B's sizes: 20.3 against 21.5 at 8 rows, 19.5 against 22.4 at 16 and 17, 20.2 against 27 at 32,
    23.4 against 30.7 at 64; Qwen3-8B's 36.7 against 37.8, 35.9 against 38.0, 34.4 against 52, 38.2 against 52.7. At 65 to 96
    rows against the kernel whose waves own rows of x (Qwen3-4B's 23.7 to 26.3 against 26.0 to 28.3, Qwen3-8B's 39 to 40.5
    against 44 to 48) and the library (2 x 17,408 of 5,120, 340 MiB: 79.9 / 84.3 / 89.8 against 95.0 / 93.4 / 98.4 at 65 / 80 /
    96 rows; 2 x 25,600 of 5,120, 500 MiB: 106.9 / 110.5 / 118.9 against 108.8 / 109.8 / 113.8, left to the library)."""
    m, k = x.shape
    return (m <= WIDE_ROWS or (m <= ops.PANEL_ROWS and w_gate_up.numel() * w_gate_up.element_size() <= _PANEL_BYTES)) and \
        k % ops.PANEL_GROUP == 0 and few_rows_ok(x, w_gate_up) and within_direct_reach(x, w_gate_up)


_PANEL_BYTES = 384 << 20        # gate/up matrices up to here go there at 65 to 96 rows too
_TALL_SWIGLU_BYTES = 256 << 20  # gate/up matrices up to here go to the kernel whose waves own rows of x beyond that, up to 256 rows


def tall_swiglu_ok(x: torch.Tensor, w_gate_up: torch.Tensor) -> bool:
    """Does the fused gate/up product with its activation go, at 97 to 256 rows, and at 65 to 96 where ``panel_swiglu_ok``, which is
    asked first, leaves it (K a multiple of 64 alone), to the kernel whose waves each own
    rows of x? In-graph times on rotating cold weights, us, against the vendor library plus the activation kernel:
    Qwen3-4B's sizes 30.0 against 35.6 at 128 rows, 36.3 against 51.0 at 256; Qwen3-8B's 46.8 against 55.5 and 57.9
    against 66.1; Qwen3-14B's (356 MB) 102 against 100 and 129 against 111, so matrices beyond 256 MiB stay with the
    library."""
    m, k = x.shape
    return WIDE_ROWS < m <= ops.TALL_ROWS and k % ops.TALL_GROUP == 0 and few_rows_ok(x, w_gate_up) and \
        within_direct_reach(x, w_gate_up) and w_gate_up.numel() * w_gate_up.element_size() <= _TALL_SWIGLU_BYTES


_MANY_TILE = (256, 128)         # rows and outputs of a workgroup of gemm_many_glu; one runs on a compute unit
_MANY_FILLED = 0.89
_MANY_DEPTHS = (1536, 3072)
_MANY_FLOPS = 1.1e12


def _many_glu_pays(m: int, n: int, k: int) -> bool:
    """Is the fused gate/up product of many rows ahead of the vendor library's product and the activation kernel, whether
    ``library_tuning`` has chosen the library's kernels or not? Where its rounds of workgroups are nearly full. A full round
    keeps up with the library's best (1.3 to 1.4 PFLOP/s) and saves the activation's pass, some 11 us a round; places of the
    last round that stay empty, and rows of a tile that are not there, cost as much as filled ones, where the library goes to
    smaller tiles. Time against the library's, as it comes / tuned, product and activation in a chain on rotating weights, 199
    sizes: with 0.89 to 1 of the rounds filled 0.94 / 0.97 on average (0.68 to 1.03 / 0.84 to 1.05), from 0.85 on 0.96 / 0.99
    (up to 1.03), from 0.74 on 1.01 / 1.01 (up to 1.10), from 0.6 on 1.08 / 1.06. Whole steps of 12 layers of Qwen3-4B (2 x
    9,728 of 2,560): 2,560 rows 0.868 / 0.987, 5,099 0.932 / 0.992, 6,144 0.959 / 1.006, 8,192 0.953 / 0.995, 9,472 0.955 /
    0.985, 10,752 0.978 / 0.999, 768 0.987 / 0.986, 1,536 0.999 / 0.991 of the time; left to the library: 1,188 rows 1.044 /
    1.034, 1,368 1.010 / 1.021, 2,126 1.012 / 1.013, and 2,048 0.963 / 1.020 (0.79 filled).
    Beyond 1.1e12 operations the library takes them: 12,806 rows are 0.992 / 0.996 on one card and up to 1.02 on others, 13,824
    0.999 / 0.995, 16,384 1.009 / 1.006, 20,480 0.978 / 0.983, 32,000 1.019 / 1.016.
    The depths are those at which this holds. At K = 1,024 filling and draining a tile takes a quarter of its time
    (Qwen3-0.6B, full rounds, whole steps: 0.995 to 1.006 / 1.008 to 1.024); at K = 4,096 the activation is a tenth of the
    product and the library reaches 1.5 PFLOP/s (Qwen3-8B likewise: 0.958 to 1.002 / 1.012 to 1.023)."""
    rows, outputs = _MANY_TILE
    rounds = -(-(-(-m // rows) * -(-n // outputs)) // _COMPUTE_UNITS)
    return _MANY_DEPTHS[0] <= k <= _MANY_DEPTHS[1] and 4.0 * m * n * k <= _MANY_FLOPS and \
        m * n >= _MANY_FILLED * rounds * _COMPUTE_UNITS * rows * outputs


def many_glu_ok(x: torch.Tensor, w_gate_up: torch.Tensor) -> bool:
    """``_many_glu_pays``, and the operands suit the kernel."""
    m, k = x.shape
    return m > ops.TALL_ROWS and k % ops.MANY_STEP == 0 and few_rows_ok(x, w_gate_up) and \
        within_direct_reach(x, w_gate_up) and _many_glu_pays(m, w_gate_up.shape[0] // 2, k)


def within_direct_reach(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Do both operands lie within what the kernels that bring them straight into LDS can address (32-bit byte
    offsets from the operand's start)? Larger ones go to the kernels that hold 64-bit addresses."""
    return w.numel() * w.element_size() < ops.DIRECT_REACH and \
        x.shape[0] * x.stride(0) * x.element_size() < ops.DIRECT_REACH


def linear(x: torch.Tensor, w: torch.Tensor, *, out_dtype: torch.dtype | None = None, allow_partials: bool = False,
           partial_rows: int | None = None):
    """Returns ``[rows, out]`` in ``out_dtype`` (default: the dtype of ``x``), or, where the caller allows it and a
    split of K pays, ``Partials`` (``partial_rows``: only for steps of at most so many rows; one, whole, where the kernel
    splits K over the waves of a workgroup alone)."""
    m, k = x.shape
    if partial_rows is not None and m > partial_rows:
        allow_partials = False
    n = w.shape[0]
    out_dtype = out_dtype or x.dtype
    if x.dtype == torch.float32:
        if ops.lines_ok(x, w) and lines_pay_f32(m, n, k):
            return ops.gemm_rows_f32(x, w, torch.empty((m, n), dtype=torch.float32, device=x.device))
        if m <= STREAM_ROWS and ops.rows_f32_ok(x, w):
            splits = rows_f32_splits(n, k) if allow_partials else 1
            if splits > 1:
                partials = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
                return Partials(ops.gemm_rows_f32(x, w, partials, splits), splits)
            product = ops.gemm_stream_f32 if streams_f32(m, n, k) else ops.gemm_rows_f32
            return product(x, w, torch.empty((m, n), dtype=torch.float32, device=x.device))
        out = torch.empty((m, n), dtype=torch.float32, device=x.device)
        if m <= STREAM_ROWS and k % 4 == 0 and w.data_ptr() % 16 == 0:
            return ops.gemm_stream_f32(x, w, out)         # rows of x at any address: that kernel reads them value by value
        if ops.rows_f32_ok(x, w):
            if ops.direct_f32_ok(x, w):
                return ops.gemm_direct_f32(x, w, out)
            return ops.gemm_block_f32(x, w, out, shape=0)
        return ops.gemm_tiled(x, w, out)
    few_ok = few_rows_ok(x, w)
    if out_dtype == torch.float32 and not allow_partials and m > STREAM_ROWS and n <= ops.NARROW_OUTPUTS and few_ok:
        return ops.gemm_narrow_bf16(x, w, torch.empty((m, n), dtype=torch.float32, device=x.device))
    library_ok = k % 8 == 0 and n % 8 == 0 and x.is_contiguous() and out_dtype == x.dtype
    if m <= STREAM_ROWS and few_ok:
        splits, group, depth = stream_plan(n, k, allow_partials)
        if lines_pay(m, n, k, splits > 1):
            # whole sums; unrounded where the other kernel would have left partial ones
            if splits > 1:
                return Partials(ops.gemm_lines(x, w, torch.empty((m, n), dtype=torch.float32, device=x.device))[None], 1)
            return ops.gemm_lines(x, w, torch.empty((m, n), dtype=out_dtype, device=x.device))
        if splits > 1:
            partials = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
            ops.gemm_stream_bf16(x, w, None, partials, group, splits, depth)
            return Partials(partials, splits)
        out = torch.empty((m, n), dtype=out_dtype, device=x.device)
        ops.gemm_stream_bf16(x, w, out, None, group, 1, depth)
        return out
    if m <= ops.MID_ROWS and (allow_partials or out_dtype == torch.float32) and few_ok and k % ops.MID_GROUP == 0 and \
            within_direct_reach(x, w) and mid_pays(m, n, k, allow_partials):
        waves, splits = mid_plan(m, n, k, allow_partials)
        partials = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
        ops.gemm_mid_bf16(x, w, partials, splits, waves)
        return Partials(partials, splits) if allow_partials else partials[0]
    if m <= WIDE_ROWS and few_ok:
        splits, group, depth = wide_plan(n, k, allow_partials)
        if splits > 1:
            partials = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
            ops.gemm_wide_bf16(x, w, None, partials, group, splits, depth)
            return Partials(partials, splits)
        if not library_ok:
            out = torch.empty((m, n), dtype=out_dtype, device=x.device)
            ops.gemm_wide_bf16(x, w, out, None, group, 1, depth)
            return out
    if m <= ops.TALL_ROWS and allow_partials and few_ok and k % ops.TALL_GROUP == 0 and within_direct_reach(x, w):
        tiles, splits = tall_plan(m, n, k)
        partials = torch.empty((splits, m, n), dtype=torch.float32, device=x.device)
        ops.gemm_tall_bf16(x, w, partials, splits, tiles)
        return Partials(partials, splits)
    if library_ok:
        return torch.mm(x, w.t())
    out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    if few_ok:
        return ops.gemm_block_bf16(x, w, out)
    return ops.gemm_tiled(x, w, out)


def linears(x: torch.Tensor, products: list) -> list:
    """``linear(x, w, out_dtype=dtype)`` for every ``(w, dtype)`` of ``products`` (``dtype`` None: that of ``x``): in one launch
    for few rows whose products go to the kernel of whole lines anyway, alone and as one matrix."""
    m, k = x.shape
    if together_pay(x, [w for w, _ in products]):
        outs = [torch.empty((m, w.shape[0]), dtype=dtype or x.dtype, device=x.device) for w, dtype in products]
        ops.gemm_lines_beside(x, [(w, out) for (w, _), out in zip(products, outs)])
        return outs
    return [linear(x, w, out_dtype=dtype) for w, dtype in products]


def together_pay(x: torch.Tensor, weights: list) -> bool:
    m, k = x.shape
    return x.dtype == torch.bfloat16 and 1 < len(weights) <= ops.LINES_TOGETHER and \
        all(ops.lines_ok(x, w) and lines_pay(m, w.shape[0], k) for w in weights) and lines_pay(m, sum(w.shape[0] for w in weights), k)


@contextlib.contextmanager
def library_tuning():
    """While open, the vendor library times its candidate kernels for every product shape it meets for the
    first time and keeps the fastest; afterwards those shapes use what was kept and nothing more is timed.

    The reference plans the same kind of choice, measured on the real GPU before the timed region
    (AGENTS.md:567). It is torch's TunableOp; what it finds is written to a file in the temporary folder
    when the process ends, never to the working directory. Not to be open while a graph is captured.
    """
    import torch.cuda.tunable as tunable
    if not tunable.is_enabled():
        tunable.set_filename(os.path.join(tempfile.gettempdir(), f"dryft_amd-products-{os.getpid()}.csv"))
        tunable.enable(True)
    tunable.tuning_enable(True)
    try:
        yield
    finally:
        tunable.tuning_enable(False)
