"""Where the planners' rules change: segment lengths by size, and whole blocks of rows in the matrix-core tiles."""
import numpy as np
import pytest

from georefine_amd import _fused


@pytest.mark.parametrize("rows,cols,segment", [
    (256, 512, 16), (3839, 1024, 16), (3840, 1024, 32),          # 15 * 2^18 weights
    (900, 4096, 16), (256, 4112, 16), (900, 4160, 32),           # rows longer than 4096: 32 where it divides, else 16
    (2252, 5120, 32), (2253, 5120, 64), (1023, 8192, 32),        # 11 * 2^20
    (1024, 8192, 32), (1024, 8256, 64), (1010, 8256, 32),        # rows longer than 8192: 2^23
    (4096, 4096, 64), (9000, 1040, 16),                          # what divides the row comes first
])
def test_segment_length_by_size(rows, cols, segment):
    assert _fused.choose_segment(cols, rows=rows) == segment
    assert _fused.choose_segment(cols, 16, rows=rows) == 16  # a caller's choice stands


@pytest.mark.parametrize("rows,cols,asked,segment", [
    (300, 1024, 64, 64), (300, 1056, 64, 32), (300, 1040, 64, 16), (300, 1152, 256, 32), (17408, 1152, 256, 64),
    (300, 1088, 128, 32), (2000, 5280, 64, 32), (300, 144, 48, 48), (300, 1024, 8, 32), (17408, 1024, 8, 64),
])
def test_a_caller_that_asks_for_a_length_does_not_get_the_smallest_matrices_index(rows, cols, asked, segment):
    assert _fused.choose_segment(cols, asked, rows=rows) == segment


@pytest.mark.parametrize("class_rows,spr,whole", [
    ([64] * 16, 160, True),     # sixteen waves, one workgroup a compute unit
    ([16] * 15 + [17], 35, True),  # two a unit, 17 tiles for 512 slots
    ([188] * 16, 96, False),    # two a unit, 384 tiles of 512 and more: spread
])
def test_row_blocks_stay_whole_where_workgroups_do_not_share_a_unit(class_rows, spr, whole):
    table = 36 * 1024
    lds = lambda p, r, cap: table + _fused.gemm_shape(p, r)[2] // 64 * 16 * cap
    threads, p, r, n_slabs, tiles, cap, lds_bytes, k = _fused.choose_gemm_tiling(
        spr, np.array(class_rows), lambda lanes: 208, lds, seg_len=32, table_bytes=table, split=True)
    assert threads == _fused.gemm_shape(p, r)[2] and tiles == sum(-(-c // r) for c in class_rows) * k
    assert (r % 16 == 0) == whole


def _predictive_plan(rows, cols, symbols=130):
    """A plan as a predictive frame has it (16 labels, 16 bins), without the frame."""
    from georefine_amd import bitexact_predictive_gpu as gpu
    rng = np.random.default_rng(rows)
    seg = gpu._fused_segment((rows, cols))
    freq = np.zeros((256, 2048), dtype=np.uint32)
    for c in range(256):
        f = np.exp(-0.5 * ((np.arange(symbols) - rng.uniform(20, symbols - 20)) / 8) ** 2) + 1e-5
        f = np.maximum(1, (f / f.sum() * 65536).astype(np.int64))
        f[np.argmax(f)] += 65536 - f.sum()
        freq[c, 300:300 + symbols] = f
    labels = np.sort(rng.integers(0, 16, rows)).astype(np.uint8)
    n = rows * cols // seg
    offsets = 4 + np.arange(n, dtype=np.int64) * seg * 3 // 8 + rng.integers(0, 4, n)
    return freq, _fused.FramePlan((rows, cols), 16, 16, labels, freq, np.full(n, 1 << 23, dtype=np.uint32), offsets,
                                  int(offsets[-1]) + 40, seg, image=gpu._word_image, lut_budget=gpu._LUT_BUDGET)


@pytest.mark.parametrize("rows,cols,both", [(4096, 4096, True), (8192, 4096, True), (2048, 4096, False), (1024, 1024, False),
                                            (9000, 1024, False)])
def test_vector_alu_launches_take_the_smaller_lookups_where_those_are_faster(rows, cols, both):
    from georefine_amd import bitexact_predictive_gpu as gpu
    freq, plan = _predictive_plan(rows, cols)
    walk = plan.for_vector_alus(freq, gpu._WALK_LUT_BUDGET, gpu._word_image)
    assert (walk is not plan) == both and plan.lognb == 12
    if both:
        assert walk.lognb == 11 and walk.lut.shape == (16, 16 << 11) and plan.lut.shape == (16, 16 << 12)
        assert np.array_equal(walk.lut, _fused.sparse_tables(freq, 16, 16, 5, gpu._word_image)[0])
        tall, fine = (p.tiling(1, waves=True) for p in (plan, walk))
        assert tall["scalars"]["n_tiles"] <= 256 < fine["scalars"]["n_tiles"] and 2 * fine["lds"] <= _fused.MAX_LDS
        assert fine["lds"] == _fused.lds_bytes_waves(16, 11, walk.tabn, 2, *(fine["scalars"][k] for k in (
            "threads", "lanes_per_row", "rows_per_tile", "n_slabs", "piece_cap")))
    assert plan.for_vector_alus(freq, gpu._LUT_BUDGET, gpu._word_image) is plan  # nothing smaller asked for


@pytest.mark.parametrize("rows,cols,smaller", [(4096, 4096, True), (8192, 2048, True), (5120, 5120, False), (2048, 2048, False),
                                               (2048, 8192, False)])
def test_matrix_core_launches_take_smaller_lookups_where_three_workgroups_share_a_unit(rows, cols, smaller):
    from georefine_amd import bitexact_predictive_gpu as gpu
    freq, plan = _predictive_plan(rows, cols)
    matrix = plan.for_matrix_cores(freq, gpu._MATRIX_LUT_BUDGET, gpu._word_image)
    assert (matrix is not plan) == smaller and plan.lognb == 12
    if smaller:
        assert matrix.lognb == 10 and np.array_equal(matrix.lut, _fused.sparse_tables(freq, 16, 16, 6, gpu._word_image)[0])
        tall, fine = plan.gemm_tiling(), matrix.gemm_tiling()
        assert tall["scalars"]["n_tiles"] <= 256 < fine["scalars"]["n_tiles"] and 3 * fine["lds"] <= _fused.MAX_LDS
        assert fine["scalars"]["threads"] <= 640 and 0 < plan.gemm_share(tall) < matrix.gemm_share(fine) <= 1
    assert plan.for_matrix_cores(freq, gpu._LUT_BUDGET, gpu._word_image) is plan  # nothing smaller asked for


@pytest.mark.parametrize("class_rows,spr,seg,fitted", [
    ([320] * 16, 96, 64, True),     # 5120 x 6144: ten of sixteen rows a tile in 512 tiles, or whole blocks in 480
    ([64] * 16, 160, 32, True),     # 1024 x 5120
    ([320] * 16, 272, 64, False),   # 5120 x 17408: the two models agree
    ([312] * 15 + [320], 48, 32, False),  # 5000 x 1536: faster at many rows, slower at few
])
def test_fitted_gemm_tilings_only_where_every_row_count_gains(class_rows, spr, seg, fitted):
    table = 35456
    lds = lambda p, r, cap, unit: max(table + _fused.gemm_shape(p, r)[2] // 64 * (unit or 16 * cap),
                                      _fused.gemm_shape(p, r)[2] // 64 * 4096)
    args = (spr, np.array(class_rows), lambda lanes: 240 if seg == 64 else 112, lds)
    plan = lambda f: _fused.plan_gemm_tiling(*args, seg_len=seg, table_bytes=table, split=True, fitted=f,
                                             unit_fn=lambda: 2832 if seg == 64 else 16 * 112)
    plain, other = plan(False), plan(True)
    assert (other != plain) == fitted
    times = []
    for threads, p, r, n_slabs, tiles, _, lds_bytes, k, _ in (plain, other):
        assert threads == _fused.gemm_shape(p, r)[2] and n_slabs == -(-spr // p) and lds_bytes <= _fused.MAX_LDS
        assert tiles == sum(-(-c // r) for c in class_rows) * k and k <= n_slabs
        taller = r > 16
        blocks = sum(-(-c // 16) for c in class_rows) * k / tiles if taller else 1.0
        times.append(_fused.gemm_times(*(np.array([v]) for v in (threads, -(-r // 16), blocks, n_slabs, tiles, k, lds_bytes)),
                                       spr, seg, table)[:, 0])
    assert np.all(times[0] >= 1.04 * times[1]) if fitted else plain == other


@pytest.mark.parametrize("rows,cols,lines", [(5120, 6144, True), (9000, 2048, False), (1024, 5120, None)])
def test_whole_lines_where_sixteen_waves_a_unit_are_enough(rows, cols, lines):
    rng = np.random.default_rng(rows)
    seg = 64 if lines is not None else 32
    n = rows * cols // seg
    offsets = 4 + np.arange(n, dtype=np.int64) * seg * 9 // 16 + rng.integers(0, 4, n)
    plan = _fused.FramePlan((rows, cols), 16, 4, (np.arange(rows) % 16).astype(np.uint8), np.tile(
        np.r_[np.full(64, 1024), np.zeros(192)].astype(np.uint32), (64, 1)), np.full(n, 1 << 23, dtype=np.uint32), offsets,
        int(offsets[-1]) + 64, seg)
    tiling = plan.lines_tiling()
    assert (tiling is not None) == bool(lines)
    if lines:
        g = tiling["scalars"]
        assert g["threads"] in (512, 1024) and sorted(tiling["tile_rows"][tiling["tile_rows"] < rows]) == list(range(rows))
        assert tiling["lds"] * (1024 // g["threads"]) <= _fused.MAX_LDS


@pytest.mark.parametrize("rows,cols,other", [(1024, 4096, True), (2048, 2048, False), (5120, 5120, False)])
def test_predictive_products_take_the_fitted_tiling_where_it_is_sure(rows, cols, other):
    from georefine_amd import bitexact_predictive_gpu as gpu
    _, plan = _predictive_plan(rows, cols)
    plain, fitted = plan.gemm_tiling(), plan.gemm_tiling(True)
    assert (plain["scalars"] != fitted["scalars"]) == other and fitted["lds"] <= _fused.MAX_LDS
    g = fitted["scalars"]
    tiles = fitted["tile_rows"].reshape(-1, g["rows_per_tile"])
    assert sorted(tiles[tiles < rows].tolist()) == list(range(rows)) and g["n_tiles"] == len(tiles) * g["k_parts"]
    assert g["threads"] == _fused.gemm_shape(g["lanes_per_row"], g["rows_per_tile"])[2]


def test_a_matrix_core_tiling_is_planned_once_for_a_plan_and_anew_for_other_lookups_and_settings(monkeypatch):
    from georefine_amd import bitexact_predictive_gpu as gpu
    freq, plan = _predictive_plan(1024, 4096)
    plain, fitted = plan.gemm_tiling(), plan.gemm_tiling(True)
    assert plan.gemm_tiling() is plain and plan.gemm_tiling(False) is plain and plan.gemm_tiling(True) is fitted is not plain
    other = plan.with_lookups(freq, gpu._MATRIX_LUT_BUDGET, gpu._word_image).gemm_tiling()
    assert other is not plain and other["lds"] != plain["lds"] and plan.gemm_tiling() is plain
    monkeypatch.setenv("GEOREFINE_FUSED_GEMM_TILING", "16,16,1")
    assert plan.gemm_tiling()["scalars"]["lanes_per_row"] == 16
    monkeypatch.delenv("GEOREFINE_FUSED_GEMM_TILING")
    monkeypatch.setattr(_fused, "GEMM_SPLIT", False)
    assert plan.gemm_tiling(True)["scalars"]["k_parts"] == 1 < fitted["scalars"]["k_parts"]
