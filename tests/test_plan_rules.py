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
