"""Which form of the MFMA kernels a grouped GEMM takes, and how those for few rows per expert are launched (host code only, no GPU)."""
import pytest
import torch

from flux_amd import capi

BF16, F16, FP8 = torch.bfloat16, torch.float16, torch.float8_e4m3fn


@pytest.mark.parametrize("dtype,block_scaled,line", [(BF16, False, 32), (F16, False, 32), (FP8, False, 24), (FP8, True, 24)])
def test_form_by_rows(dtype, block_scaled, line):
    k = 4096 if dtype == FP8 else 2048  # rows of 4 KiB and many columns: the streaming form's up to 16 rows per expert

    def form(rows, splits=None):
        return capi.gemm_launch_info(dtype, 8, rows, 16384, k, block_scaled=block_scaled, splits=splits).form

    def panel(rows):
        return capi.gemm_launch_info(dtype, 8, rows, 16384, k, block_scaled=block_scaled, panel=True)

    assert form(1) == form(32) == capi.GEMM_STREAM  # no expert can have more than one chunk of 32 rows
    assert form(33) == form(128) == capi.GEMM_BY_SPLITS and panel(33).cols == panel(128).cols == 0
    assert form(129) == form(768) == capi.GEMM_BY_SPLITS and panel(129).cols > 0 and panel(768).cols > 0
    assert form(769) == form(100000) == capi.GEMM_MACRO_TILES
    # up to `line` rows per expert both forms for few rows take a launch, with the same sums over K
    assert [panel(rows).sums for rows in (129, 8 * line, 8 * line + 1, 768)] == [4, 4, 1, 1]
    # under 16 experts with rows: one chunk each
    assert form(80, [32, 0, 10, 0, 0, 30, 8, 0]) == capi.GEMM_STREAM
    assert form(80, [33, 0, 10, 0, 0, 29, 8, 0]) == capi.GEMM_MACRO_TILES
    assert form(80, [80, -5, 0, 0, 0, 0, 0, 0]) == capi.GEMM_MACRO_TILES
    # counts past max_rows do not exist
    assert form(40, [20, 20, 400, 0, 0, 0, 0, 0]) == capi.GEMM_STREAM

    # from 16 on a quarter more chunks of 32 rows than experts with rows
    def form_of(splits):
        return capi.gemm_launch_info(dtype, len(splits), 200, 16384, k, block_scaled=block_scaled, splits=splits).form

    assert form_of([33] * 4 + [0] * 5 + [3] * 12) == form_of([129] + [0] * 5 + [3] * 15) == capi.GEMM_STREAM
    assert form_of([33] * 5 + [0] * 5 + [2] * 11) == form_of([129, 33] + [0] * 5 + [2] * 14) == capi.GEMM_MACRO_TILES
    assert form_of([33] + [0] * 5 + [3] * 14) == capi.GEMM_MACRO_TILES  # 15 experts with rows


@pytest.mark.parametrize("dtype,splits,n,k,form,without", [
    (BF16, [0, 0, 0, 240, 0, 0, 0, 0], 1024, 2048, capi.GEMM_PANEL, capi.GEMM_PANEL),  # small weights: whatever the splits
    (BF16, [60] * 4 + [0] * 4, 14336, 4096, capi.GEMM_PANEL, capi.GEMM_BY_SPLITS),
    (BF16, [40, 40, 20, 20, 10, 10, 10, 10], 14336, 4096, capi.GEMM_PANEL, capi.GEMM_BY_SPLITS),
    (F16, [100] + [20] * 7, 14336, 4096, capi.GEMM_PANEL, capi.GEMM_BY_SPLITS),
    (F16, [240] + [0] * 7, 14336, 4096, capi.GEMM_MACRO_TILES, capi.GEMM_BY_SPLITS),
    (FP8, [66, 66] + [13] * 14, 4096, 4096, capi.GEMM_MACRO_TILES, capi.GEMM_BY_SPLITS),
    (FP8, [66] + [13] * 15, 4096, 4096, capi.GEMM_PANEL, capi.GEMM_BY_SPLITS),
    (BF16, [129] + [90] * 7, 14336, 4096, capi.GEMM_PANEL, capi.GEMM_BY_SPLITS),
    (BF16, [400] + [50] * 7, 14336, 4096, capi.GEMM_MACRO_TILES, capi.GEMM_BY_SPLITS),
    (BF16, [120] * 8, 14336, 4096, capi.GEMM_MACRO_TILES, capi.GEMM_MACRO_TILES)])
def test_form_is_that_of_the_kernel_that_computes(dtype, splits, n, k, form, without):
    info = capi.gemm_launch_info(dtype, len(splits), sum(splits), n, k, splits=splits)
    panel = capi.gemm_launch_info(dtype, len(splits), sum(splits), n, k, splits=splits, panel=True)
    assert info.form == form and panel.computes == (form == capi.GEMM_PANEL)
    assert capi.gemm_launch_info(dtype, len(splits), sum(splits), n, k).form == without
    assert (panel.cols > 0) == (form == capi.GEMM_PANEL or without == capi.GEMM_BY_SPLITS)
    assert (info.stream_cols, info.stream_waves, info.stream_workgroups, info.stream_lds_bytes) == (0, 0, 0, 0)


def test_generic_shapes_have_no_streaming_form():
    assert capi.gemm_launch_info(BF16, 8, 16, 4096, 1023).form == capi.GEMM_GENERIC
    with pytest.raises(RuntimeError, match="cu_count"):
        capi.gemm_launch_info(BF16, 8, 16, 4096, 1024, cu_count=0)
    with pytest.raises(RuntimeError, match="ngroups"):
        capi.gemm_launch_info(BF16, 8, 16, 4096, 1024, ngroups=5)


@pytest.mark.parametrize("dtype", [BF16, F16, FP8])
@pytest.mark.parametrize("experts,rows,n,k", [(8, 74, 2048, 4096), (8, 20, 2048, 8192), (64, 90, 400, 8192), (1, 8, 16384, 8192), (16, 200, 1408, 2048),
                                              (64, 576, 1408, 2048), (64, 576, 1408, 4096), (32, 256, 2048, 2048), (64, 1500, 1408, 2048)])
def test_weight_groups_do_not_change_how_k_is_split(dtype, experts, rows, n, k):
    """A launch of several weight groups adds K up in the order of a launch per group: as many waves, or sums of the panel tiles, and the
    same choice between these forms and the macro tiles."""
    def split(groups):
        info, panel = (capi.gemm_launch_info(dtype, experts, rows, n, k, ngroups=groups, panel=p) for p in (False, True))
        return (panel.sums if panel.cols else info.stream_waves, info.form == capi.GEMM_BY_SPLITS, panel.chunk_rows if panel.cols else 32)

    assert split(2) == split(3) == split(4) == split(1)


@pytest.mark.parametrize("dtype,block_scaled", [(BF16, False), (FP8, False), (FP8, True)])
@pytest.mark.parametrize("experts,rows,n,k", [(8, 16, 4224, 2064 - 16), (8, 180, 14336, 4096), (32, 400, 7168, 2048), (4, 8, 1024, 8192)])
@pytest.mark.parametrize("margin", [1, 100, 249, 255, 1000])
def test_margin_leaves_whole_compute_units(dtype, block_scaled, experts, rows, n, k, margin):
    """With a margin every workgroup has a compute unit for itself (more than half of its 160 KiB of LDS), and there are no more
    of them than units that may be used."""
    def launch(margin):
        info, panel = (capi.gemm_launch_info(dtype, experts, rows, n, k, block_scaled=block_scaled, cu_margin=margin, panel=p) for p in (False, True))
        if panel.cols > 0:
            return panel.workgroups, panel.lds_bytes, (info.form, panel.cols, panel.sums)
        return info.stream_workgroups, info.stream_lds_bytes, (info.form, info.stream_cols, info.stream_waves)

    workgroups, lds_bytes, form = launch(margin)
    assert 80 * 1024 < lds_bytes <= 160 * 1024
    assert 1 <= workgroups <= max(1, 256 - margin)
    assert launch(0)[2] == form  # same bits


@pytest.mark.parametrize("dtype,k,block_scaled", [(BF16, 8, False), (FP8, 16, False), (FP8, 128, True)])
@pytest.mark.parametrize("groups", [1, 4])
def test_a_launch_stays_below_the_grid_limit(dtype, k, block_scaled, groups):
    """2^32 threads are more than a launch may have: workgroups then walk the items.  Beyond what an int numbers the macro tiles run."""
    if block_scaled and groups > 1:
        return
    for experts, n in ((1024, 1 << 18), (1024, 1 << 20), (700, (1 << 20) + 4), (4, 1 << 24)):
        info = capi.gemm_launch_info(dtype, experts, experts, n, k, ngroups=groups, block_scaled=block_scaled)
        assert info.form in (capi.GEMM_STREAM, capi.GEMM_BY_SPLITS)
        assert 1 <= info.stream_workgroups <= ((1 << 32) - 1) // (info.stream_waves * 64)
    assert capi.gemm_launch_info(dtype, 1024, 1024, 1 << 20, k, block_scaled=block_scaled).stream_workgroups == 256
    assert capi.gemm_launch_info(dtype, 1024, 1024, 1 << 24, k, block_scaled=block_scaled).form == capi.GEMM_MACRO_TILES
    assert capi.gemm_launch_info(dtype, 1024, 1024, 1 << 24, k, block_scaled=block_scaled, panel=True).cols == 0


@pytest.mark.parametrize("dtype,experts,n,k,most", [(BF16, 64, 512, 1024, 128), (BF16, 128, 256, 1024, 128), (FP8, 16, 2048, 2048, 128),
                                                     (BF16, 48, 512, 1024, 170), (BF16, 8, 2048, 2048, 192), (FP8, 2, 8192, 4096, 192)])
def test_small_weights_many_rows_are_panel_tiles_while_one_expert_is_one_round(dtype, experts, n, k, most):
    """These launches run the panel tiles whatever the splits; with more than 96 rows per expert only while 512 workgroups of 64 columns and
    128 rows compute them all, also if one expert has every row."""
    form = [capi.gemm_launch_info(dtype, experts, rows * experts, n, k).form for rows in (96, most, most + 1)]
    assert form == [capi.GEMM_PANEL, capi.GEMM_PANEL, capi.GEMM_MACRO_TILES]
    assert (most * experts + 127) // 128 * (n // 64) <= 512 and (most == 192 or (most + 1) * experts / 128 * (n // 64) > 512)


@pytest.mark.parametrize("dtype,experts,rows,n,k,forms", [
    (FP8, 16, 60, 2048, 2048, "PSSS"), (FP8, 16, 20, 2048, 2048, "PPPP"), (BF16, 64, 44, 512, 1024, "PSSS"), (BF16, 8, 60, 1024, 2048, "PPSS"),
    (BF16, 32, 128, 512, 1024, "PPMM"), (BF16, 8, 150, 1024, 2048, "PPMM")])
def test_small_launches_count_all_weight_groups(dtype, experts, rows, n, k, forms):
    """P: panel tiles whatever the splits, S: the splits decide, M: macro tiles, for 1 to 4 weight groups; with few rows per expert the
    groups do not choose."""
    names = {capi.GEMM_PANEL: "P", capi.GEMM_BY_SPLITS: "S", capi.GEMM_MACRO_TILES: "M"}
    assert "".join(names[capi.gemm_launch_info(dtype, experts, rows * experts, n, k, ngroups=g).form] for g in (1, 2, 3, 4)) == forms


@pytest.mark.parametrize("dtype,experts,rows,n,k,ngroups,block_scaled,panel", [
    (FP8, 16, 64, 4096, 2560, 1, False, True), (FP8, 16, 65, 4096, 2560, 1, False, False), (FP8, 16, 96, 2048, 2560, 1, False, True),
    (FP8, 16, 96, 2176, 2560, 1, False, False), (FP8, 16, 80, 2048, 2048, 2, False, False), (FP8, 16, 80, 4096, 6144, 1, False, True),
    (FP8, 32, 80, 4096, 2560, 1, False, True),  # 256 columns
    (FP8, 16, 80, 4096, 2560, 1, True, True), (BF16, 16, 80, 4096, 2560, 1, False, True)])
def test_fp8_short_k_in_several_rounds_is_for_the_macro_tiles(dtype, experts, rows, n, k, ngroups, block_scaled, panel):
    got = capi.gemm_launch_info(dtype, experts, experts * rows, n, k, ngroups=ngroups, block_scaled=block_scaled, panel=True)
    form = capi.gemm_launch_info(dtype, experts, experts * rows, n, k, ngroups=ngroups, block_scaled=block_scaled).form
    assert (got.cols > 0) == panel and form == (capi.GEMM_BY_SPLITS if panel else capi.GEMM_MACRO_TILES)


@pytest.mark.parametrize("block_scaled,splits,n,k,form", [
    (True, [129] + [54] * 31, 2048, 7168, capi.GEMM_MACRO_TILES), (True, [128] + [54] * 31, 2048, 7168, capi.GEMM_PANEL),  # 528 items and 512
    (True, [129] * 2 + [50] * 30, 2560, 2560, capi.GEMM_PANEL), (True, [129] + [55] * 15, 4096, 5120, capi.GEMM_MACRO_TILES),  # 680 and 544
    (True, [129] + [60] * 15, 2048, 4096, capi.GEMM_PANEL),  # 272: the first round and the second
    (True, [129] * 2 + [60] * 23 + [0] * 7, 2560, 4096, capi.GEMM_MACRO_TILES),  # 540, of experts with rows 500; one busy expert less 520, 480
    (True, [129] + [60] * 23 + [0] * 8, 2560, 4096, capi.GEMM_PANEL), (True, [129] + [60] * 24 + [0] * 7, 2560, 4096, capi.GEMM_MACRO_TILES),
    (False, [129] + [54] * 31, 2048, 7168, capi.GEMM_PANEL)])
def test_block_scaled_extra_chunks_take_no_extra_round(block_scaled, splits, n, k, form):
    """Block-scaled panel tiles of 128 rows and columns, one workgroup to each of 256 units: experts of several chunks must fit the rounds
    that one chunk each would take, from two on."""
    rows = max(sum(splits), 41 * len(splits))
    info = capi.gemm_launch_info(FP8, len(splits), rows, n, k, splits=splits, block_scaled=block_scaled)
    panel = capi.gemm_launch_info(FP8, len(splits), rows, n, k, splits=splits, block_scaled=block_scaled, panel=True)
    assert (panel.cols, panel.chunk_rows) == (128, 128)
    assert info.form == form and panel.computes == (form == capi.GEMM_PANEL)


@pytest.mark.parametrize("dtype", [BF16, F16, FP8])
@pytest.mark.parametrize("experts,rows,k", [(64, 64 * 64, 8), (1024, 1024 * 64, 8), (8, 8 * 90, 16)])
def test_panel_tiles_of_256_columns_have_a_workgroup_per_item(dtype, experts, rows, k):
    """That kernel computes one item per workgroup: where a launch cannot have that many, other tiles, which walk, take it."""
    def info(n):
        return capi.gemm_launch_info(dtype, experts, rows, n, k * (2 if dtype == FP8 else 1), panel=True)

    for n in (2048 * 256, 1 << 21, 1 << 23, 1 << 25, 30000000, 1 << 28):
        got = info(n)
        if got.cols == 256:
            assert got.workgroups >= experts * ((n + 255) // 256)
        assert got.cols == 0 or 1 <= got.workgroups <= ((1 << 31) - 1) // 256
    if (experts, dtype) == (64, BF16):  # 73 chunks of 128 rows at most: both sides of 2^31 threads
        below, above = info(114912 * 256), info(114912 * 256 + 4)
        assert (below.cols, below.workgroups) == (256, 73 * 114912)
        assert (above.cols, above.workgroups) == (128, 256)


# dual32: the same with fp32 results
@pytest.mark.parametrize("dtype,experts,rows,n,k,block_scaled,dual,dual32", [
    (BF16, 8, 320, 14336, 4096, False, True, True), (BF16, 8, 321, 14336, 4096, False, False, False), (F16, 8, 512, 4096, 3072, False, False, False),
    (F16, 8, 512, 4096, 3008, False, True, True), (F16, 8, 513, 4096, 3008, False, False, False), (F16, 64, 1536, 2048, 1408, False, True, False),
    (F16, 64, 1536, 1408, 2048, False, False, False), (BF16, 64, 768, 1408, 1984, False, True, False), (BF16, 64, 769, 1408, 1984, False, False, False),
    (BF16, 64, 1024, 2048, 1472, False, True, True), (BF16, 64, 1025, 2048, 1472, False, True, False), (F16, 64, 1500, 2048, 960, False, True, True),
    (F16, 64, 1501, 2048, 960, False, True, False), (BF16, 64, 4000, 2048, 448, False, True, True),
    (FP8, 32, 512, 2048, 7168, False, True, True), (FP8, 32, 513, 2048, 7168, False, False, False), (FP8, 32, 1024, 2048, 3072, False, True, False),
    (FP8, 32, 1024, 2048, 2944, False, True, True), (FP8, 32, 1025, 2048, 2944, False, True, False), (FP8, 32, 1500, 2048, 1920, False, True, True),
    (FP8, 32, 1501, 2048, 1920, False, True, False), (FP8, 32, 4000, 2048, 896, False, True, True),
    (FP8, 32, 4000, 7168, 2944, False, True, False), (FP8, 32, 4000, 7168, 7168, True, True, True),
    # not whole steps of K, one step, columns that are not in eights, too many experts
    (BF16, 8, 300, 4096, 4104, False, False, False), (FP8, 8, 300, 4096, 128, True, False, False), (BF16, 8, 300, 4100, 4096, False, False, True),
    (FP8, 129, 300, 512, 512, True, False, False)])
def test_dual_tiles_by_rows_and_k(dtype, experts, rows, n, k, block_scaled, dual, dual32):
    def is_dual(**kw):
        return capi.gemm_dual_tiles(dtype, experts, rows * experts, n, k, block_scaled=block_scaled, **kw)

    assert capi.gemm_launch_info(dtype, experts, rows * experts, n, k, block_scaled=block_scaled).form == capi.GEMM_MACRO_TILES
    assert is_dual() == is_dual(gathered=True) == dual
    assert is_dual(d_fp32=True) == is_dual(d_fp32=True, gathered=True) == dual32
    for flag in (capi.SCHED_HALF_LINE_FILLS, capi.SCHED_WHOLE_LINE_FILLS):
        assert is_dual(sched_flags=flag) == (dual and block_scaled)


@pytest.mark.parametrize("experts,rows,n,k,dual", [
    # up to 128 tiles whatever the splits: macro tiles up to 64 rows
    (1, 59, 416, 13056, False), (1, 64, 416, 256, False), (1, 65, 416, 13056, True), (3, 45, 272, 7168, False), (64, 64, 264, 256, True),
    (8, 64, 3064, 512, False), (8, 64, 3336, 512, True),
    # more than 256: macro tiles up to 448 and 64 rows, and up to 96 rows with K of 4 KiB and more
    (64, 64, 1032, 256, False), (64, 64, 1544, 256, True), (64, 64, 1544, 4096, False), (64, 65, 1032, 2048, True), (64, 96, 1032, 4096, False),
    (64, 96, 1032, 3968, True), (64, 97, 1032, 4096, True),
    # columns in 64s: the panel tiles take them, and what is left by splits stays with the dual tiles
    (64, 64, 4096, 4096, True)])
def test_block_scaled_launches_of_few_rows_run_the_macro_tiles(experts, rows, n, k, dual):
    kind = capi.gemm_launch_info(FP8, experts, rows * experts, n, k, block_scaled=True).form
    assert kind == (capi.GEMM_MACRO_TILES if n % 64 else capi.GEMM_BY_SPLITS)
    for d_fp32 in (False, True):
        assert capi.gemm_dual_tiles(FP8, experts, rows * experts, n, k, block_scaled=True, d_fp32=d_fp32) == dual


@pytest.mark.parametrize("dtype,block_scaled", [(BF16, False), (F16, False), (FP8, False), (FP8, True)])
@pytest.mark.parametrize("experts,rows,n,kbytes,dual", [  # dual: None for "but for block scales"
    # up to 128 columns, rows of K of 1 KiB and more or block scales: macro tiles up to 128 tiles whatever the splits; up to 256 with 4 KiB (1 KiB) and more
    (5, 300, 32, 2048, False), (5, 300, 128, 1024, False), (5, 300, 128, 896, None), (5, 300, 136, 2048, True),
    (64, 256, 128, 2048, False), (64, 260, 128, 2048, None), (64, 260, 128, 4096, False), (64, 260, 128, 3968, None), (64, 260, 128, 896, True),
    (100, 500, 128, 4096, True)])
def test_few_tiles_of_few_columns_run_the_macro_tiles(dtype, block_scaled, experts, rows, n, kbytes, dual):
    k = kbytes // (1 if dtype == FP8 else 2)
    assert capi.gemm_launch_info(dtype, experts, rows * experts, n, k, block_scaled=block_scaled).form == capi.GEMM_MACRO_TILES
    for d_fp32 in (False, True):
        assert capi.gemm_dual_tiles(dtype, experts, rows * experts, n, k, block_scaled=block_scaled, d_fp32=d_fp32) == (not block_scaled if dual is None else dual)
