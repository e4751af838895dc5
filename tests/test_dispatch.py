"""Which matrix-product kernel a shape goes to, decided on the host: checked here with tensors that have shapes but
no storage."""

import pytest
import torch


def fake(rows, cols, dtype=torch.bfloat16):
    return torch.empty((rows, cols), dtype=dtype, device="meta")


def test_operands_beyond_32_bit_offsets_stay_away_from_the_direct_to_lds_kernels():
    """The kernels that bring their operands straight into LDS address them by 32-bit byte offsets and refuse more;
    the dispatch must not send them such operands (every step of up to 64 or 256 rows would fail)."""
    from dryft_amd.csrc import ops
    from dryft_amd.parts.linear import panel_swiglu_ok, within_direct_reach
    x = fake(8, 16384)
    assert panel_swiglu_ok(x, fake(2 * 25600, 16384))                  # 1.7 GB: within reach
    big = fake(2 * 70000, 16384)                                       # 4.6 GB of weights
    assert big.numel() * 2 >= ops.DIRECT_REACH
    assert not panel_swiglu_ok(x, big) and not within_direct_reach(x, big)
    assert within_direct_reach(fake(256, 16384), fake(5120, 16384))
    wide_rows = torch.empty((200, 16), dtype=torch.bfloat16, device="meta").as_strided((200, 16), (1 << 24, 1))
    assert not within_direct_reach(wide_rows, fake(64, 16))            # rows 32 MB apart: the activations are out of reach


def test_plans_split_k_only_where_partial_sums_are_taken():
    from dryft_amd.parts.linear import small_mid_plan, stream_plan, tall_plan, wide_plan
    # 33 to 64 rows: one workgroup of 64 outputs a compute unit, and no run of K left empty
    assert small_mid_plan(6144, 2560) == 2 and small_mid_plan(2560, 4096) == 6 and small_mid_plan(2560, 9728) == 6
    assert small_mid_plan(5120, 25600) == 1 and small_mid_plan(64, 64) == 1          # beyond 48 MiB; one group of K
    assert stream_plan(6144, 2560, may_split=False)[0] == 1
    assert stream_plan(2560, 9728, may_split=True)[0] > 1
    assert wide_plan(6144, 2560, may_split=False)[0] == 1
    assert wide_plan(2560, 4096, may_split=True)[0] > 1
    # 65 to 256 rows: a split that leaves no run of K empty, tile counts the kernel has, about one workgroup a
    # compute unit where the shape allows it; a single group of K cannot be split
    from dryft_amd.csrc import ops
    for n, k in ((6144, 2560), (2560, 9728), (5120, 17408), (1024, 2048), (80, 64), (100, 192)):
        for m in (65, 128, 129, 256):
            tiles, splits = tall_plan(m, n, k)
            assert 4 <= tiles <= 8 and ops.gemm_mid_splits(k, splits) == splits
    assert tall_plan(256, 80, 64) == (4, 1)
    tiles, splits = tall_plan(256, 2560, 9728)
    assert 200 <= -(-2560 // (16 * tiles)) * splits <= 256


def test_gate_up_kernel_by_rows_and_size():
    from dryft_amd.parts.linear import panel_swiglu_ok, tall_swiglu_ok
    fake = lambda rows, cols: torch.empty((rows, cols), dtype=torch.bfloat16, device="meta")
    w = fake(2 * 9728, 2560)
    assert panel_swiglu_ok(fake(64, 2560), w) and not tall_swiglu_ok(fake(64, 2560), w)
    assert tall_swiglu_ok(fake(65, 2560), w) and tall_swiglu_ok(fake(256, 2560), w) and not tall_swiglu_ok(fake(257, 2560), w)
    assert not tall_swiglu_ok(fake(128, 5120), fake(2 * 17408, 5120))           # beyond 256 MiB: the vendor library
    assert not tall_swiglu_ok(fake(128, 2592), fake(512, 2592))                 # K no multiple of 64


@pytest.mark.parametrize("rows,k,offset,stride,want", [(3, 64, 0, 64, "few"), (3, 64, 1, 64, "gemm_stream_f32"), (3, 64, 0, 67, "gemm_stream_f32"),
                                                       (16, 36, 3, 39, "gemm_stream_f32"), (3, 66, 0, 66, "gemm_tiled"),
                                                       (17, 64, 1, 64, "gemm_tiled"), (17, 64, 0, 64, "gemm_direct_f32"),
                                                       (17, 36, 0, 36, "gemm_block_f32")])
def test_float32_products_by_where_the_rows_lie(monkeypatch, rows, k, offset, stride, want):
    """Up to 16 rows that do not start at 16-byte addresses go to the kernel that reads them value by value."""
    from dryft_amd.csrc import ops
    from dryft_amd.parts import linear as linear_module
    called = []
    for name in ("gemm_rows_f32", "gemm_stream_f32", "gemm_direct_f32", "gemm_block_f32", "gemm_tiled"):
        monkeypatch.setattr(ops, name, lambda x, w, out, *a, name=name, **b: called.append(name) or out)
    held = torch.empty(rows * stride + 8)
    first = (-held.data_ptr() % 16) // 4 + offset
    x = held[first:].as_strided((rows, k), (stride, 1))
    w = torch.empty(40 * k + 4)
    w = w[(-w.data_ptr() % 16) // 4:][:40 * k].view(40, k)
    linear_module.linear(x, w)
    assert called in ([want], ["gemm_rows_f32" if want == "few" else want])


@pytest.mark.parametrize("rows,outputs", [(2_097_120, 64), (2_097_121, 32), (4_194_241, 64), (5_000_000, 64), (8_388_480, 64)])
def test_float32_blocks_of_many_rows_fit_a_grid(rows, outputs):
    """The block that the library chooses has no more than 65,535 blocks of rows as long as one of the three has."""
    from dryft_amd.csrc import ops
    shape = ops._fn("gemm_f32", "dryft_gemm_direct_f32_shape")(rows, outputs)
    assert -(-rows // (128, 64, 32)[shape]) <= 65535


@pytest.mark.parametrize("rows,outputs,depth,ours", [
    (1188, 9728, 2560, False), (1368, 9728, 2560, False), (2126, 9728, 2560, False), (2842, 9728, 2560, False),
    (2048, 6144, 2048, False), (3072, 6144, 2048, False), (1557, 8192, 2048, False), (2150, 3072, 1024, False), (4360, 3072, 1024, False),
    (1530, 12288, 4096, False), (6144, 12288, 4096, False), (12806, 12288, 4096, False),
    (16384, 9728, 2560, False), (32000, 9728, 2560, False), (12806, 9728, 2560, False), (10752, 9728, 2560, True),
    (768, 9728, 2560, True), (2560, 9728, 2560, True), (4096, 9728, 2560, True), (5099, 9728, 2560, True), (8192, 9728, 2560, True),
    (1280, 6144, 2048, True), (1024, 8192, 2048, True), (5099, 8192, 2048, True), (8447, 8960, 1536, True)])
def test_gate_up_of_many_rows_goes_where_it_was_measured_ahead(rows, outputs, depth, ours):
    """Rounds of tiles that are nearly full stay here, at sizes beyond 2.5e11 operations too; sizes that were 1 to 10 % slower
    than the vendor library, as it comes or tuned, go there."""
    from dryft_amd.parts.linear import many_glu_ok
    assert many_glu_ok(fake(rows, depth), fake(2 * outputs, depth)) == ours


@pytest.mark.parametrize("rows,heads,kv,size,longest,keys,form", [
    (1, 16, 8, 128, 1, 20, "rows"), (4, 16, 8, 128, 1, 4096, "rows"), (64, 32, 8, 128, 1, 280, "rows"),       # decoding
    (16, 16, 8, 128, 16, 200, "rows"), (5, 32, 8, 128, 5, 4096, "rows"), (17, 16, 8, 128, 17, 17, "tiles"),   # steps of few rows
    (33, 16, 8, 128, 33, 4096, "tiles"), (525, 16, 8, 128, 253, 253, "tiles"), (20, 32, 8, 128, 5, 64, "tiles"),
    (1, 32, 1, 128, 1, 150, "plain"), (8, 32, 1, 128, 1, 512, "plain"), (1, 32, 1, 128, 1, 1024, "rows"), (16, 32, 1, 128, 1, 64, "rows"),
    (1, 8, 1, 256, 1, 150, "plain"), (17, 8, 1, 256, 17, 17, "plain"), (1, 8, 1, 256, 1, 512, "rows"), (40, 8, 1, 256, 40, 40, "tiles"),
    (4, 16, 4, 192, 1, 150, "plain"), (4, 16, 8, 256, 1, 150, "rows"), (5, 16, 8, 256, 5, 200, "rows")])
def test_float32_attention_goes_where_it_was_measured_ahead(rows, heads, kv, size, longest, keys, form):
    from dryft_amd.parts.attention import float32_form
    assert float32_form(rows, heads, kv, size, longest, keys) == form


def test_every_entry_point_is_called_with_as_many_arguments_as_it_declares():
    """The table of ctypes signatures against the ``extern "C"`` declarations in the HIP sources: every entry point the
    Python side calls exists in its library's source and takes as many arguments as the table lists."""
    import os
    import re

    from dryft_amd.csrc import ops
    folder = os.path.dirname(os.path.abspath(ops.__file__))
    for module, functions in ops._SIGNATURES.items():
        with open(os.path.join(folder, module + ".hip")) as f:
            text = f.read()
        declared = {m.group(1): m.group(2) for m in re.finditer(r"DRYFT_API\s+\w+\s+(\w+)\s*\(([^)]*)\)", text)}
        for name, signature in functions.items():
            assert name in declared, f"{module}.hip declares no {name}"
            count = len([a for a in declared[name].split(",") if a.strip()])
            assert count == len(signature), f"{name}: declared with {count} arguments, called with {len(signature)}"


@pytest.mark.parametrize("rows", [17, 32, 33, 64, 65, 96, 97, 128])
@pytest.mark.parametrize("n,k", [(6144, 2560), (2560, 9728), (1024, 64), (5120, 17408), (151936, 1024), (96, 4096)])
def test_products_of_17_to_128_rows_fill_the_units_once(rows, n, k):
    """A plan that splits K leaves no run empty and needs one round of workgroups; a whole product has one run."""
    from dryft_amd.csrc import ops
    from dryft_amd.parts.linear import mid_plan
    waves, splits = mid_plan(rows, n, k, True)
    assert waves in ops.MID_WAVES and ops.gemm_mid_splits(k, splits) == splits
    assert splits == 1 or -(-n // (16 * waves)) * splits <= 256
    assert mid_plan(rows, n, k, False)[1] == 1


@pytest.mark.parametrize("rows,experts,top,k,gated,kernel", [
    (1, 16, 4, 2048, True, 1), (4, 16, 4, 512, False, 1), (4, 16, 4, 256, True, 1), (4, 16, 4, 248, True, 0), (4, 16, 4, 504, False, 0),
    (4, 16, 4, 520, False, 0), (4, 16, 4, 1032, False, 0), (4, 16, 4, 1032, True, 1), (4, 16, 4, 824, True, 0), (5, 16, 4, 504, True, 0), (5, 16, 4, 512, True, 1), (8, 16, 4, 768, False, 0),
    (8, 2, 2, 1024, False, 1), (16, 16, 4, 1024, False, 1), (16, 16, 4, 1024, True, 1), (9, 4, 2, 1024, True, 2), (9, 4, 2, 960, True, 0), (9, 4, 2, 1040, True, 0),
    (9, 4, 2, 2048, False, 0), (8, 4, 4, 960, True, 1), (16, 4, 4, 136, False, 0)])
def test_experts_of_few_rows_go_where_they_were_measured_ahead(rows, experts, top, k, gated, kernel):
    """By rows, places an expert and K; what was up to 2.4 times slower through the kernel of whole lines goes to the other one."""
    from dryft_amd.csrc import ops
    plan = ops.MoePlan(rows * top, experts, "cpu", most_places=rows)
    assert ops.moe_lines_pay(plan, experts, k, gated) == kernel


@pytest.mark.parametrize("rows,size,taps,takes", [
    (16, 128, 4, True), (16, 256, 4, False), (16, 160, 4, False), (17, 256, 4, True), (17, 288, 4, False), (4, 48, 4, False), (16, 32, 4, True),
    (2, 32, 8, True), (3, 32, 8, False), (128, 32, 5, False), (8, 64, 8, True), (9, 64, 8, False), (17, 64, 8, True), (16, 96, 16, True)])
def test_one_row_of_a_gated_recurrence_goes_where_it_was_measured_ahead(rows, size, taps, takes):
    from dryft_amd.csrc import ops
    blocks = 3
    aligned = lambda *shape, dtype: torch.empty(shape, dtype=dtype)
    proj, state = aligned(rows, 2 * blocks * size, dtype=torch.bfloat16), aligned(rows, blocks * size, dtype=torch.float32)
    gate, vector = aligned(blocks, size, size, dtype=torch.bfloat16), aligned(blocks * size, dtype=torch.float32)
    assert ops.rglru_token_takes(proj, state, gate, gate, (vector,) * 4, blocks, taps) == takes
    assert not ops.rglru_token_takes(proj.float(), state, gate, gate, (vector,) * 4, blocks, taps)


@pytest.mark.parametrize("seqs,rows,width,kv_keys,spares,takes", [
    (4, 8, 64, 4000, False, True), (4, 9, 64, 4000, False, False), (4, 8, 128, 4000, True, True), (4, 8, 128, 4000, False, False),
    (4, 7, 128, 4000, False, True), (31, 7, 160, 4000, True, True), (4, 8, 160, 4000, True, False), (4, 4, 144, 4000, False, True),
    (4, 5, 144, 4000, True, False), (4, 1, 176, 100, True, False), (1, 1, 192, 100, False, False), (8, 2, 256, 100, True, False),
    (32, 16, 128, 1 << 20, False, True), (32, 16, 256, 1 << 20, False, True), (32, 16, 192, 4687, False, True),
    (32, 16, 192, 4688, True, False), (64, 17, 64, 100, True, False)])
def test_the_turn_goes_into_attention_where_it_was_measured_ahead(seqs, rows, width, kv_keys, spares, takes):
    """Heads of 192 features and 5 to 8 rows a kv head of odd widths were up to a third slower in one launch."""
    from dryft_amd.csrc import ops
    assert ops.turns_in_attention(seqs, rows, width, kv_keys, spares) == takes


@pytest.mark.parametrize("rows,heads,kv,keys,width,splits", [
    (4, 16, 8, 512, 128, 8), (4, 16, 8, 128, 64, 1), (4, 16, 8, 192, 64, 3), (4, 16, 1, 304, 256, 1), (4, 64, 4, 334, 256, 1),
    (4, 16, 1, 4096, 256, 32), (8, 64, 4, 158, 80, 1), (1, 6, 2, 114, 256, 1), (1, 4, 1, 1024, 192, 16), (1, 16, 1, 256, 80, 1)])
def test_float32_keys_are_split_where_that_was_measured_ahead(rows, heads, kv, keys, width, splits):
    """What was up to twice as slow split, since the last workgroup adds up many wide parts, stays with one workgroup."""
    from dryft_amd.parts.attention import float32_splits
    assert float32_splits(rows, heads, kv, keys, width) == splits


@pytest.mark.parametrize("rows,n,k,split,pays", [
    (17, 5120, 25600, True, True), (64, 5120, 25600, True, True), (65, 5120, 25600, True, False), (128, 5120, 17408, True, True),
    (65, 10240, 9856, True, False), (65, 10240, 9792, True, True), (96, 1024, 2048, True, True), (97, 1024, 2048, True, False),
    (97, 4096, 2048, True, True), (97, 4096, 1984, True, False), (128, 151936, 2560, False, True)])
def test_products_of_17_to_128_rows_by_size(rows, n, k, split, pays):
    """Split products leave for the kernel whose waves own rows of x beyond 64 rows and 192 MiB, and beyond 96 rows below 16 MiB."""
    from dryft_amd.parts.linear import mid_pays
    assert mid_pays(rows, n, k, split) == pays


@pytest.mark.parametrize("rows,outputs,k,kernel", [
    (64, 9728, 2560, "panel"), (65, 9728, 2560, "panel"), (96, 9728, 2560, "panel"), (97, 9728, 2560, "tall"), (256, 9728, 2560, "tall"),
    (257, 9728, 2560, "library"), (64, 25600, 5120, "panel"), (96, 17408, 5120, "panel"), (65, 25600, 5120, "library"),
    (97, 17408, 5120, "library"), (65, 19661, 5120, "library"), (65, 19660, 5120, "panel"), (65, 512, 2624, "tall"), (64, 512, 2624, "library")])
def test_gate_up_by_rows_size_and_depth(monkeypatch, rows, outputs, k, kernel):
    """In the order in which the feed-forward asks: what it calls."""
    from dryft_amd.csrc import ops
    from dryft_amd.parts import mlp
    called = []
    for name, what in (("gemm_few_glu_bf16", "few"), ("gemm_panel_swiglu_bf16", "panel"), ("gemm_tall_swiglu_bf16", "tall"),
                       ("gemm_many_glu_bf16", "many"), ("silu_mul", "library")):
        monkeypatch.setattr(ops, name, lambda *a, what=what, **b: called.append(what))
    monkeypatch.setattr(mlp, "linear", lambda x, w, **kw: x)
    part = mlp.SwiGLU(k, outputs)
    part.w_gate_up, part.w_down = fake(2 * outputs, k), fake(k, outputs)
    part.forward(fake(rows, k), None, leave_product=True)
    assert called == [kernel]


@pytest.mark.parametrize("file,define,constant,more", [
    ("token_step.h", "TOKEN_MAX_DIM", "TOKEN_MAX_DIM", 0), ("rglru.hip", "RG_TOKEN_BLOCK", "RGLRU_TOKEN_BLOCK", 0),
    ("rglru.hip", "RG_MAX_TAPS", "RGLRU_MAX_TAPS", 0), ("attn_f32.hip", "F32_MAX_SPLITS", "ATTN_F32_SPLITS", 0),
    ("gemm_lines.hip", "LINES_BESIDE", "LINES_TOGETHER", 1), ("gemm.hip", "PANEL_ROWS", "PANEL_ROWS", 0),
    ("gemm.hip", "PANEL_GROUP", "PANEL_GROUP", 0), ("gemm.hip", "MID_GROUP", "MID_GROUP", 0), ("gemm.hip", "MID_ROWS", "MID_ROWS", 0), ("mlstm.hip", "MLSTM_COLS", "MLSTM_COLUMNS", 0),
    ("conv.hip", "CONV_MAX_TAPS", "CONV_MAX_TAPS", 0), ("ssm.hip", "SSM_MAX_STATE", "SSM_MAX_STATE", 0),
    ("moe.hip", "MOE_MAX_EXPERTS", "MOE_MAX_EXPERTS", 0)])
def test_limits_that_both_sides_hold_are_the_same(file, define, constant, more):
    import os
    import re

    from dryft_amd.csrc import ops
    with open(os.path.join(os.path.dirname(os.path.abspath(ops.__file__)), file)) as f:
        value = re.search(rf"^#define {define} (\d+)", f.read(), re.M)
    assert value and int(value.group(1)) + more == getattr(ops, constant)
