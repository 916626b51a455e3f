"""decode() through wave units at the edges of the quad exchange: rows whose segments do not fill a
quad, segments of 16 and 32 words, tiles with empty slots, one row, one segment."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [3, 67, 130])
@pytest.mark.parametrize("cols,segment", [(64, 64), (64 * 5, 64), (64 * 33, 64), (32 * 7, 32), (16 * 9, 16), (96, 48), (128 * 3, 128)])
def test_wave_units_store_every_word(rows, cols, segment):
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd import bitexact_predictive_codec as predictive
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    from georefine_amd.bitexact_predictive_gpu import HipPredictiveTensor
    rng = np.random.default_rng(rows * 131 + cols)
    # (few distinct exponents, and one class where 64 contexts' tables would outgrow the words, so that
    # even the smallest frame is coded and not raw words)
    words = (rng.choice([0x3C00, 0x3C20, 0x3D00], (rows, cols)) | rng.integers(0, 32, (rows, cols))
             | rng.integers(0, 2, (rows, cols)) << 15).astype(np.uint16)
    frame = codec.encode(words)
    if rows * cols < 1000:
        frame = codec.encode(words, row_classes=1, col_classes=1)
    assert frame[5] != 1
    t = HipContextTensor(frame, fused_segment=segment)
    assert t.fused is not None and t.fused_plan["seg_len"] == segment and t._store_tiling()[3]["scheme"] == 1
    guard = torch.full((rows * cols + 64,), 0x5A5A, device="cuda", dtype=torch.int16)  # what the launch must not touch
    t._launch(t._lib.grf_bctx_fused_decode, t.fused, t._store_tiling()[0], guard.data_ptr(), t.error.data_ptr())
    got = guard.cpu().numpy().view(np.uint16)
    assert np.array_equal(got[:rows * cols].reshape(words.shape), words) and (got[rows * cols:] == 0x5A5A).all()
    assert np.array_equal(t.decode().view(torch.int16).cpu().numpy().view(np.uint16), words)
    if segment % 32 == 0:
        p = HipPredictiveTensor(predictive.encode(words, words ^ np.uint16(1)), words ^ np.uint16(1), fused_segment=segment)
        assert (p.fused is None) == (p.mode == 2)  # (a handful of words is kept raw)
        if p.fused is not None:
            assert np.array_equal(p.decode(None).view(torch.int16).cpu().numpy().view(np.uint16), words)


@pytest.mark.parametrize("first", [0, 1, 2, 4, 7])
@pytest.mark.parametrize("cols,segment", [(64 * 5, 64), (16 * 9, 16), (32 * 7, 32)])
def test_output_begins_at_any_word(cols, segment, first):
    """The C entry points store to a caller's buffer from any word on, by the wave units and by
    slab tilings, and touch nothing on either side."""
    import ctypes
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd import bitexact_predictive_codec as predictive
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    from georefine_amd.bitexact_predictive_gpu import HipPredictiveTensor
    rng = np.random.default_rng(cols)
    words = (rng.choice([0x3C00, 0x3C20, 0x3D00], (67, cols)) | rng.integers(0, 32, (67, cols))).astype(np.uint16)
    t = HipContextTensor(codec.encode(words), fused_segment=segment)
    assert t.fused is not None
    stream = torch.cuda.current_stream().cuda_stream
    launches = [(t._lib.grf_bctx_fused_decode, t, (), t._tiling(1)), (t._lib.grf_bctx_fused_decode, t, (), t._tiling(0))]
    if segment % 32 == 0:
        p = HipPredictiveTensor(predictive.encode(words, words ^ np.uint16(1)), words ^ np.uint16(1), fused_segment=segment)
        assert p.fused is not None
        bins = (p.buffers["context_bins"].data_ptr(),)
        launches += [(p._lib.grf_ppcx_fused_decode, p, bins, p._tiling_for("waves")),
                     (p._lib.grf_ppcx_fused_decode, p, bins, p._tiling_for(0))]
    for fn, tensor, extra, (tiling, _, _, scalars) in launches:
        guard = torch.full((first + words.size + 64,), 0x5A5A, device="cuda", dtype=torch.int16)
        tensor.error.zero_()
        status = fn(ctypes.byref(tensor.fused), ctypes.byref(tiling), *extra, guard.data_ptr() + 2 * first,
                    tensor.error.data_ptr(), stream)
        assert status == 0 and tensor.error.item() == 0
        got = guard.cpu().numpy().view(np.uint16)
        assert np.array_equal(got[first:first + words.size].reshape(words.shape), words), scalars["scheme"]
        assert (got[:first] == 0x5A5A).all() and (got[first + words.size:] == 0x5A5A).all()


@pytest.mark.parametrize("cols,segment", [(64 * 65, 64), (16 * 9, 16), (32 * 64, 32), (64 * 2, 64)])
def test_row_gather_clamps_rejects_and_reports(cols, segment):
    """Ids outside the matrix: an IndexError, or clamped where the caller vouches for them; a
    miss is reported to the call that checks and only there; waves without segments."""
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    rng = np.random.default_rng(cols)
    words = (rng.choice([0x3C00, 0x3C20, 0x3D00], (70, cols)) | rng.integers(0, 32, (70, cols))).astype(np.uint16)
    t = HipContextTensor(codec.encode(words), fused_segment=segment)
    assert t.fused is not None
    ids = torch.tensor([[-5, 0, 69], [70, 3, 1 << 40]])
    got = t.gather_rows(ids, check=False, validate=False).view(torch.int16).cpu().numpy().view(np.uint16)
    assert np.array_equal(got, words[ids.clamp(0, 69).numpy()])
    for bad in (70, -1, 1 << 32):
        with pytest.raises(IndexError):
            t.gather_rows(torch.tensor([1, bad]))
    assert np.array_equal(t.gather_rows(torch.tensor([1]).cuda()).view(torch.int16).cpu().numpy().view(np.uint16), words[[1]])
    t.buffers["fused_seg_state"].view(torch.int32)[t.index_slot(7, 1)] += 1  # forced from the host; kernels finish normally
    t.gather_rows(torch.tensor([7]), check=False)
    assert t.error.item() != 0
    t.gather_rows(torch.tensor([8]))
    assert t.error.item() == 0
    with pytest.raises(codec.CodecError):
        t.gather_rows(torch.tensor([7]))
    assert t.error.item() != 0


@pytest.mark.parametrize("cols,segment", [(64 * 65, 64), (16 * 9, 16), (32 * 7, 32)])
def test_gather_by_a_tiling_of_the_callers(cols, segment):
    """grf_bctx_fused_gather, for callers of the C interface that name the rows in a slab tiling: any
    order, a row twice, an empty slot, which leaves its output as it was."""
    import ctypes
    import torch
    from georefine_amd import _fused, _hip_abi
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    rng = np.random.default_rng(cols)
    words = (rng.choice([0x3C00, 0x3C20, 0x3D00], (70, cols)) | rng.integers(0, 32, (70, cols))).astype(np.uint16)
    t = HipContextTensor(codec.encode(words), fused_segment=segment)
    assert t.fused is not None
    rows = np.array([69, 3, 3, 0xFFFFFFFF, 0, 41], dtype=np.uint32)
    classes = np.array([t._plan.row_class[r] if r < 70 else 0 for r in rows], dtype=np.uint8)
    spr = cols // segment
    lanes = min(spr, 64)
    scalars = dict(threads=64, lanes_per_row=lanes, rows_per_tile=1, n_slabs=-(-spr // lanes), n_tiles=len(rows),
                   piece_cap=t._plan._cap(lanes), scheme=_fused.SCHEME_SLABS, k_parts=0)
    block, position, _ = t._plan.residual_order()
    _fused.validate_host(t._plan, dict(scalars=scalars, tile_rows=rows, tile_class=classes), "gather", row_pos=position, block=block)
    on_device = torch.from_numpy(rows.view(np.int32)).cuda(), torch.from_numpy(classes).cuda()
    g = _hip_abi.GrfFusedTiling()
    g.tile_rows, g.tile_class = (a.data_ptr() for a in on_device)
    for key, value in scalars.items():
        setattr(g, key, value)
    out = torch.full((len(rows) + 1, cols), 0x5A5A, device="cuda", dtype=torch.int16)
    t._launch(t._lib.grf_bctx_fused_gather, ctypes.byref(t.fused), ctypes.byref(g), out.data_ptr(), t.error.data_ptr())
    got = out.cpu().numpy().view(np.uint16)
    for j, row in enumerate(rows):
        assert np.array_equal(got[j], words[row] if row < 70 else np.full(cols, 0x5A5A, dtype=np.uint16)), j
    assert (got[-1] == 0x5A5A).all() and t.error.item() == 0


def test_row_gather_when_another_thread_took_the_last_word(monkeypatch):
    """The words that gathers report to are shared by threads: a list that was not empty a moment ago
    is no row outside the matrix."""
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd import bitexact_context_gpu as gpu
    rng = np.random.default_rng(5)
    words = (rng.choice([0x3C00, 0x3C20, 0x3D00], (70, 128)) | rng.integers(0, 32, (70, 128))).astype(np.uint16)
    t = gpu.HipContextTensor(codec.encode(words))

    class Taken(list):  # looks as it did before the other thread's turn
        def __bool__(self):
            return True

    kept = Taken()
    monkeypatch.setattr(gpu, "_host_words", kept)
    for _ in range(2):
        got = t.gather_rows(torch.tensor([3, 69]))
        assert np.array_equal(got.view(torch.int16).cpu().numpy().view(np.uint16), words[[3, 69]])
        assert len(kept) == 1 and kept[0].item() == 0  # given back, and taken the second time
