"""How many workgroups the planners let share a compute unit's LDS, which is given out in units of 1280 bytes."""
import numpy as np
import pytest

from conftest import weight_like
from georefine_amd import _fused


@pytest.mark.parametrize("lds,share", [(16, 128), (1280, 128), (1281, 64), (26880, 6), (26896, 5), (32000, 5), (32016, 4), (40960, 4),
                                       (40961, 3), (53760, 3), (53776, 2), (54608, 2), (81920, 2), (81921, 1), (163840, 1), (163841, 0)])
def test_share_of_the_units_lds(lds, share):
    assert _fused.lds_share(lds) == share
    assert _fused.lds_share(np.array([lds, 1280])).tolist() == [share, 128]


def test_three_square_siblings_reserve_what_lets_three_workgroups_share_a_unit():
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    frame = codec.encode(weight_like(np.random.default_rng(32768), 4096, 4096), residual="raw6")
    plan = HipContextTensor.host_prepare(frame, fused_segment=64)["plan"]
    tiling = _fused.plan_group([plan] * 3, gemm=True)[0]
    g = tiling["scalars"]
    assert 3 * g["n_tiles"] > 2 * 256  # (more workgroups than two a unit)
    most = _fused.GEMM_WAVES_PER_SIMD // -(-(g["threads"] // 64) // 4)
    assert most == 3 and 3 * -(-tiling["lds"] // 1280) <= 128


@pytest.mark.parametrize("lds,rounds", [(53760, 1), (54080, 2), (54613, 2)])
def test_the_models_see_the_round_that_does_not_fit(lds, rounds):
    """A wave tiling of eight waves, 768 tiles: in one round only where three share a unit."""
    tiling = dict(scalars=dict(threads=512, lanes_per_row=16, rows_per_tile=4, n_slabs=1, n_tiles=768), lds=lds)
    once = _fused.wave_time(dict(tiling, lds=50000), 64, 0)
    assert (_fused.wave_time(tiling, 64, 0) == once) == (rounds == 1)
    many = np.array([768])
    times = [_fused.gemm_times(np.array([512]), np.array([1]), np.array([1.0]), np.array([3]), many, np.array([1]), np.array([v]), 24, 64, 0)
             for v in (50000, lds)]
    assert bool((times[0] == times[1]).all()) == (rounds == 1)


@pytest.mark.parametrize("rows,siblings,spr,tiles,tight", [
    (4612, 3, 12, 480, True),    # three workgroups a unit may share: 768 slots, and 512 without the tight reservation
    (7162, 1, 22, 512, True),
    (14853, 2, 8, 512, False),   # one slab of two quads
])
def test_tiles_that_all_run_at_once_are_not_cut_shorter_to_fill_the_closer_slots(rows, siblings, spr, tiles, tight):
    table = 35200
    lds = lambda p, r, cap, unit: max(table + _fused.gemm_shape(p, r)[2] // 64 * (unit or 16 * cap), _fused.gemm_shape(p, r)[2] // 64 * 4096)
    class_rows = np.concatenate([np.bincount(np.arange(rows) % 16)] * siblings)
    found = _fused.plan_gemm_tiling(spr, class_rows, lambda lanes: 208, lds, seg_len=64, table_bytes=table, unit_fn=lambda: 2816)
    assert found[4] == tiles and (found[8] == 2816) == tight and _fused.lds_share(found[6]) >= (3 if tight else 2)
