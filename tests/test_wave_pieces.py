"""A matrix-core wave's sixteen stream pieces lie one behind the other in the LDS: what a tiling reserves
for them, and that products do not depend on where the pieces lie."""
import ctypes

import numpy as np
import pytest

from conftest import bf16_words, weight_like
from georefine_amd import _fused, _native


@pytest.mark.parametrize("rows,spr,lanes,together", [(1, 1, 4, 16), (15, 5, 4, 16), (33, 17, 4, 16), (40, 8, 3, 4), (7, 3, 64, 1)])
def test_most_units_of_consecutive_rows(rows, spr, lanes, together):
    rng = np.random.default_rng(rows * spr)
    offsets = (4 + np.cumsum(np.concatenate(([0], rng.integers(0, 60, rows * spr))))).astype(np.uint32)
    order = rng.permutation(rows).astype(np.uint32)
    flat = offsets.astype(np.int64)
    first = flat[:-1].reshape(rows, spr)[:, ::lanes]
    last = np.concatenate((first[:, 1:], flat[spr::spr][:, None]), axis=1)
    units = ((last - (first & ~15) + 8 + 15) // 16)[order]
    units = np.concatenate((np.ones((together, units.shape[1]), dtype=np.int64), units, np.ones((together, units.shape[1]), dtype=np.int64)))
    want = max(int(units[i:i + together].sum(axis=0).max()) for i in range(rows + together + 1))
    most = ctypes.c_uint32()
    call = lambda o: _native.codec().grf_unit_pieces(_native.ptr(offsets, ctypes.c_uint32), rows, spr, _native.ptr(o, ctypes.c_uint32),
                                                     lanes, together, ctypes.byref(most))
    assert call(order) == 0 and most.value == want
    order[0] = rows
    assert call(order) != 0  # a row the matrix does not have


def _tensor_plan(words, segment):
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    frame = codec.encode(words)
    return frame, HipContextTensor.host_prepare(frame, fused_segment=segment)


@pytest.mark.parametrize("rows,cols,segment", [(96, 768, 64), (37, 528, 16), (20, 2048, 256)])
def test_validator_adds_up_the_pieces_that_a_tiling_reserves_for(rows, cols, segment):
    plan = _tensor_plan(weight_like(np.random.default_rng(rows), rows, cols), segment)[1]["plan"]
    block, position, _ = plan.residual_order()
    tiling = plan.gemm_tiling()
    reserve = lambda units, use="gemm": _fused.validate_host(
        plan, dict(tiling, scalars=dict(tiling["scalars"], wave_bytes=16 * units)), use, row_pos=position, block=block)
    units = plan.quad_bytes() // 16
    assert units <= plan.quad_cap()  # (sixteen of the longest)
    reserve(units)
    held = (tiling["tile_rows"].reshape(-1, tiling["scalars"]["rows_per_tile"])[:, :16] != 0xFFFFFFFF).sum(axis=1)
    with pytest.raises(_fused.FusedUnsupported, match="the tiling reserves"):
        reserve(int(held.max()))  # a unit a row
    with pytest.raises(_fused.FusedUnsupported, match="LDS reserved"):
        reserve(160 * 64 + 1)
    gemv = plan.tiling(1, waves=True)
    with pytest.raises(_fused.FusedUnsupported, match="LDS reserved"):
        _fused.validate_host(plan, dict(gemv, scalars=dict(gemv["scalars"], wave_bytes=16 * units)), "gemv", row_pos=position, block=block)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,segment", [
    (417, 16 * 5, 16), (100, 64 * 17, 64), (257, 16 * 35, 16),  # quads without all four segments, blocks without all sixteen rows
    (20, 256 * 9, 256), (17, 512 * 9, 512),                    # pieces longer than half and than all of an instruction's 64 units
])
def test_products_do_not_depend_on_where_the_pieces_lie(rows, cols, segment):
    import torch
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    rng = np.random.default_rng(cols)
    frame, prepared = _tensor_plan(weight_like(rng, rows, cols), segment)
    t = HipContextTensor(frame, fused_segment=segment, prepared=prepared)
    assert t.fused is not None and t.fused_plan["seg_len"] == segment
    w = t.decode().double()
    g, pieces = t._gemm_tiling()[0], t._plan.quad_bytes()
    for m in (1, 20, 70):
        x = torch.from_numpy(bf16_words(rng.normal(0, 1, size=(m, cols)))).view(torch.bfloat16).cuda()
        got = []
        for reserved in (0, pieces):
            g.wave_bytes = reserved
            got.append(t.gemm(x, check=True))
        assert torch.equal(*got)
        want, scale = x.double() @ w.T, x.double().abs() @ w.abs().T
        # one rounding to BF16, and fp32 sums of at most `cols` exact products
        assert bool(((got[0].double() - want).abs() <= want.abs() * 2.0 ** -8 + scale * cols * 2.0 ** -24).all())
