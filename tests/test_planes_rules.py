"""Which matrices are held as planes, how their sums are split, and that the sizes agree with the library's (no GPU)."""
import ctypes
import re
from pathlib import Path

import numpy as np
import pytest

from georefine_amd import _fused, _hip_abi, _native, _planes
from georefine_amd import bitexact_context_codec as codec
from georefine_amd.bitexact_context_gpu import HipContextTensor

from conftest import weight_like


@pytest.mark.parametrize("rows,cols", [(1, 16), (16, 64), (17, 80), (255, 240), (1000, 256), (4097, 272), (5120, 17408), (64, 131072)])
def test_sizes_are_the_librarys_and_no_split_is_empty(rows, cols):
    lib = _native.hip()
    assert _planes.plane_bytes(rows, cols) == lib.grf_planes_bytes(rows, cols)
    assert -(-rows // 16) * _planes.visits(cols) == lib.grf_planes_visits(rows, cols)
    splits = _planes.sum_splits(rows, cols)
    each = -(-_planes.visits(cols) // splits)
    assert 1 <= splits <= 16
    assert (splits - 1) * each < _planes.visits(cols) and each <= 63


@pytest.mark.parametrize("change", [dict(splits=0), dict(splits=17), dict(splits=4), dict(cols=1028), dict(cols=1 << 18), dict(rows=0),
                                    dict(planes=8), dict(listed=None)])
def test_what_the_kernels_would_not_take_is_refused_before_a_launch(change):
    lib = _native.hip()
    good = dict(planes=4096, bases=4096, listed_at=4096, listed=4096, rows=64, cols=1024, splits=2)
    if change.get("splits") == 4:
        good.update(cols=1280)  # five visits, two a split: nothing is left for the fourth
    p = _hip_abi.GrfPlanes(**{**good, **change})
    assert lib.grf_planes_decode(ctypes.addressof(p), 4096, None) != 0 and b"grf_planes_decode" in lib.grf_last_error()
    assert lib.grf_planes_linear(ctypes.addressof(p), 4096, 2048, 1, 0, 4096, None, None, 0, None) != 0


@pytest.mark.parametrize("change", [{}, dict(splits=0), dict(splits=17), dict(rows=0), dict(cols=0), dict(planes=8), dict(listed=None)])
def test_a_workspace_is_asked_for_what_a_launch_takes_and_nothing_else(change):
    lib = _native.hip()
    p = _hip_abi.GrfPlanes(**{**dict(planes=4096, bases=4096, listed_at=4096, listed=4096, rows=5120, cols=17408, splits=12), **change})
    one = (ctypes.c_void_p * 2)(ctypes.addressof(p), None)
    for n, m, want in ((1, 1, 12 * 5120 * 4), (1, 6, 12 * 6 * 5120 * 4), (1, 128, 12 * 128 * 5120 * 4), (2, 8, 0), (2, 9, 12 * 9 * 5120 * 4)):
        assert lib.grf_planes_workspace_bytes(n, one, m) == (0 if change else want), (n, m)
    assert lib.grf_planes_workspace_bytes(2, None, 6) == 0


@pytest.mark.parametrize("rows,cols,shared", [(256, 12800, 0), (512, 12800, 0), (512, 14336, 0), (1300, 17408, 0), (1600, 17408, 0), (2400, 32768, 0),
                                              (6144, 17408, 0), (1024, 5120, 0), (512, 17408, 1), (1024, 24576, 1), (256, 32768, 1), (2048, 32768, 1),
                                              (4200, 17408, 1), (5120, 14336, 1), (5120, 17408, 1)])
def test_row_blocks_are_shared_where_that_was_measured_to_pay(rows, cols, shared):
    """One row of x: a workspace is asked for only where workgroups share row blocks (of the sizes beside own_parts)."""
    p = _hip_abi.GrfPlanes(planes=4096, bases=4096, listed_at=4096, listed=4096, rows=rows, cols=cols, splits=_planes.sum_splits(rows, cols))
    size = _native.hip().grf_planes_workspace_bytes(1, (ctypes.c_void_p * 1)(ctypes.addressof(p)), 1)
    assert (size > 0) == bool(shared)


def test_small_sparse_and_odd_frames_stay_frames():
    rng = np.random.default_rng(3)
    large = codec.encode(weight_like(rng, 512, 1024))
    few = codec.encode((rng.choice([0x3C00, 0x3C20], (4096, 1024)) | rng.integers(0, 32, (4096, 1024))).astype(np.uint16))
    assert "words" in HipContextTensor.host_prepare(large)
    for frame, how in ((codec.encode(weight_like(rng, 511, 1024)), {}), (large, {"fused": False}), (few, {"fused_segment": 64})):
        assert "words" not in HipContextTensor.host_prepare(frame, **how)


def test_the_walks_arrays_are_made_when_asked_for_and_travel():
    import pickle
    words = weight_like(np.random.default_rng(4), 512, 1040)
    prepared = HipContextTensor.host_prepare(codec.encode(words))
    assert np.array_equal(prepared["words"].reshape(words.shape), words)
    there = pickle.loads(pickle.dumps(prepared))
    for p in (prepared, there):
        assert isinstance(p["plan"], _fused.FramePlan) and p["raw6_segment"] == 16
        assert p["indexed"]["main_stream"].flags.writeable
        with pytest.raises(KeyError):
            p["no such entry"]


def test_listed_share_counts_what_is_outside_eleven_exponents():
    freq = np.zeros((2, 1024), dtype=np.uint32)  # two row classes, one column class
    freq[0, 4 * 100:4 * 111] = 1489  # eleven exponents
    freq[0, 4 * 100] += 65536 - 44 * 1489
    freq[1, 4 * 50] = freq[1, 4 * 80] = 32768
    assert _planes.listed_share(np.array([0, 0, 0, 1]), np.zeros(7, dtype=np.uint8), freq, 2, 1) == pytest.approx(0.125)


def test_plans_of_many_rows_are_what_the_launch_takes():
    lib = _native.hip()
    taken = 0
    for rows, cols, m in [(1, 16, 129), (17, 240, 2048), (300, 1040, 129), (5120, 17408, 200), (5120, 17408, 1000), (17408, 5120, 300), (64, 131072, 150),
                          (1024, 8192, 160), (65536, 512, 4000), (1 << 20, 512, 1024), (1 << 20, 512, 1025), (512, 1028, 200), (512, 1024, 128)]:
        plan = lib.grf_planes_prompt_plan(rows, cols, m)
        if cols % 8 or m <= 128 or rows * m > 1 << 30:
            assert plan == -1
        if plan < 0:
            continue
        taken += 1
        tile, parts = plan & 0xFFFF, plan >> 16
        each = -(-_planes.visits(cols) // parts)
        assert tile in (128, 256) and each <= 63 and (parts - 1) * each < _planes.visits(cols)
        assert lib.grf_planes_prompt_workspace_bytes(rows, m, plan) == (parts * m * ((rows + 3) & ~3) * 4 if parts > 1 else 0)
    assert taken >= 3


@pytest.mark.parametrize("change", [dict(plan=0), dict(plan=1 << 16 | 64), dict(plan=5 << 16 | 128), dict(plan=2 << 16 | 128), dict(ldx=1016),
                                    dict(ldx=1 << 22), dict(ldy=63), dict(y=4098), dict(x=4100), dict(m=0)])
def test_products_of_many_rows_that_a_launch_would_not_take_are_refused(change):
    lib = _native.hip()
    p = _hip_abi.GrfPlanes(planes=4096, bases=4096, listed_at=4096, listed=4096, rows=64, cols=1024, splits=2)
    a = {**dict(x=4096, ldx=1024, m=200, plan=1 << 16 | 128, y=4096, ldy=64), **change}
    assert lib.grf_planes_prompt(ctypes.addressof(p), a["x"], a["ldx"], a["m"], a["plan"], a["y"], a["ldy"], None, None, 0, None) != 0
    assert b"grf_planes_prompt" in lib.grf_last_error()


def test_assembly_that_writes_m0_says_so():
    found = 0
    for source in sorted((Path(_native.__file__).parent / "csrc").iterdir()):
        for statement in re.findall(r"\basm\b[^;]*;", source.read_text()):
            if re.search(r"\bm0\s*,", statement.split('"::')[0].replace('"m0",', "")):  # (an instruction's first operand)
                found += 1
                assert '"m0"' in statement, (source.name, statement)
    assert found >= 2
