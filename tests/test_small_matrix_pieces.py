"""Matrices with fewer rows than a matrix-core wave has slots: what the wave stages for them, empty slots
among it, against what their tilings reserve."""
import ctypes
import subprocess

import numpy as np
import pytest

from conftest import bf16_words, weight_like
from georefine_amd import _fused, _native

NONE = 0xFFFFFFFF


@pytest.fixture(scope="module")
def piece_units(tmp_path_factory):
    """The kernel's own formula, compiled for the host."""
    at = tmp_path_factory.mktemp("units")
    (at / "units.cpp").write_text(
        '#include "piece_units.h"\n'
        'extern "C" uint32_t units(int held, uint32_t first, uint32_t past) { return grf::piece_units(held != 0, first, past); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", str(_native.CSRC), str(at / "units.cpp"), "-o", str(at / "units.so")],
                   check=True)
    fn = ctypes.CDLL(str(at / "units.so")).units
    fn.argtypes, fn.restype = [ctypes.c_int, ctypes.c_uint32, ctypes.c_uint32], ctypes.c_uint32
    return fn


def _weights(rows, cols):
    rng = np.random.default_rng(rows * cols)
    target = weight_like(rng, rows, cols)
    return target, bf16_words((target.astype(np.uint32) << 16).view(np.float32) + rng.normal(0, 0.002, (rows, cols)).astype(np.float32))


def _launches(kind, rows, cols, segment):
    """(plan, tiling) of every matrix-core launch that the tensor of this matrix may make."""
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd import bitexact_predictive_codec as predictive, bitexact_predictive_gpu as gpu
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    target, ref = _weights(rows, cols)
    if kind == "bctx":
        plan = HipContextTensor.host_prepare(codec.encode(target), fused_segment=segment)["plan"]
        return [(plan, plan.gemm_tiling()), (plan, _fused.plan_group([plan], gemm=True)[0])]
    read = gpu._read_frame(predictive.encode(target, ref), ref, 256, fused=True, fused_segment=segment)
    if "fused_plan" not in read:  # (the smallest matrices are stored as they are)
        assert "raw" in read and rows * cols < 4096
        return []
    plan, matrix = read["fused_plan"], read["matrix_plan"]
    return [(matrix, matrix.gemm_tiling(matrix is plan)), (plan, _fused.plan_group([plan], gemm=True)[0])]


@pytest.mark.parametrize("rows", [*range(1, 21)])
@pytest.mark.parametrize("kind,cols,segment", [
    ("ppcx", 1536, None), ("ppcx", 4096, None), ("ppcx", 6144, None), ("ppcx", 8192, 64), ("ppcx", 2048, 128),
    ("bctx", 2048, None), ("bctx", 2048, 64), ("bctx", 8192, 64), ("bctx", 6144, 128),
])
def test_every_wave_stages_within_what_its_tiling_reserves(piece_units, kind, cols, segment, rows):
    for plan, tiling in _launches(kind, rows, cols, segment):
        g, spr = tiling["scalars"], plan.spr
        lanes, reserved = g["lanes_per_row"], (g.get("wave_bytes") or 16 * g["piece_cap"]) // 16
        block, position, held = plan.residual_order()
        offsets = _fused.order_index(plan.seg_offset, rows, spr, block, position, held)
        at = lambda q, s: int(offsets[(q - q % block) * (spr + 1) + s * block + q % block])
        most = 0
        for tile in tiling["tile_rows"].reshape(-1, g["rows_per_tile"]):
            for r0 in range(0, len(tile), 16):
                slots = [*tile[r0:r0 + 16], *[NONE] * 16][:16]
                for slab in range(0, spr, lanes):
                    for s in range(slab, min(spr, slab + lanes), 4):
                        past = min(s + 4, slab + lanes, spr)
                        # (a slot without a row is handed the empty range at the index's first entry)
                        most = max(most, sum(piece_units(0, at(0, 0), at(0, 0)) if row == NONE else
                                             piece_units(1, at(int(position[row]), s), at(int(position[row]), past)) for row in slots))
        assert most <= reserved
        _fused.validate_host(plan, tiling, "gemm", row_pos=position, block=block)
        if most > 16:  # and the validator counts no less
            with pytest.raises(_fused.FusedUnsupported, match="the tiling reserves"):
                _fused.validate_host(plan, dict(tiling, scalars=dict(g, wave_bytes=16 * (most - 1))), "gemm", row_pos=position, block=block)


def test_units_of_a_slot_at_every_phase(piece_units):
    for phase in range(16):
        assert piece_units(0, 4096 + phase, 4096 + phase) == 1
        for length in range(0, 40):
            # the aligned start to the end of the eight bytes that are read from the last byte's place on
            assert piece_units(1, 4096 + phase, 4096 + phase + length) == -(-(phase + length + 8) // 16)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,segment", [
    ("ppcx", 1, 6144, None), ("ppcx", 2, 6144, None), ("ppcx", 3, 4096, None), ("ppcx", 4, 1536, None), ("ppcx", 5, 8192, None),
    ("ppcx", 6, 1536, None), ("ppcx", 17, 1536, None), ("bctx", 2, 2048, 64), ("bctx", 2, 8192, 64), ("bctx", 5, 8192, 64),
])
def test_products_of_small_matrices(kind, rows, cols, segment):
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd import bitexact_predictive_codec as predictive
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    from georefine_amd.bitexact_predictive_gpu import HipPredictiveTensor
    target, ref = _weights(rows, cols)
    if kind == "ppcx":
        t = HipPredictiveTensor(predictive.encode(target, ref), ref, fused_segment=segment)
        product = lambda x: t.linear(None, x, check=True)
    else:
        t = HipContextTensor(codec.encode(target), fused_segment=segment)
        product = lambda x: t.gemm(x, check=True)
    assert t.fused is not None
    w = (torch.from_numpy(target.astype(np.int32)) << 16).view(torch.float32).double()
    for m in (2, 6, 20, 70):
        words = bf16_words(np.random.default_rng(m).normal(0, 1, size=(m, cols)))
        x = torch.from_numpy(words).view(torch.bfloat16)
        got, x64 = product(x.cuda()).double().cpu(), x.double()
        want, scale = x64 @ w.T, x64.abs() @ w.abs().T
        # one rounding to BF16, and fp32 sums of at most `cols` exact products
        assert bool(((got - want).abs() <= want.abs() * 2.0 ** -8 + scale * cols * 2.0 ** -24).all()), m
