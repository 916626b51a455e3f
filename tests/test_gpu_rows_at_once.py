"""Products that read several half groups of activations at once from the caller's rows: the packed copy's
bits, also where a segment is no whole number of the columns read at once, and where the matrix is too
large for more rows to be read in place."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,segment", [(50, 48 * 5, 48), (33, 32 * 7, 32), (17, 16 * 3, 16), (97, 80 * 9, 80), (5200, 8192, 64)])
@pytest.mark.parametrize("m", [1, 6, 7, 16, 17, 32])
def test_rows_read_at_once_equal_the_packed_copy(m, rows, cols, segment):
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor, PackedActivations
    rng = np.random.default_rng(7)
    words = (rng.choice([0x3C00, 0x3C20, 0x3D00], (rows, cols)) | rng.integers(0, 32, (rows, cols))).astype(np.uint16)
    key = rows, cols
    if _tensors.get("key") != key:
        _tensors.update(key=key, tensor=HipContextTensor(codec.encode(words), fused_segment=segment))
    t = _tensors["tensor"]
    assert t.fused is not None and t.fused_plan["seg_len"] == segment
    around = torch.full((m + 2, cols + 4), float("nan"), device="cuda", dtype=torch.bfloat16)
    x = around[1:m + 1, :cols]  # rows on 8-byte boundaries, with what must not be read around them
    x.copy_(torch.from_numpy(rng.standard_normal((m, cols), dtype=np.float32)))
    want = t.gemm(PackedActivations(x))
    got = torch.empty_like(want)
    g = t._gemm_tiling()[0]
    size = t._lib.grf_gemm_workspace_bytes_split(cols, rows, g.k_parts, m)
    space = torch.empty(size, device="cuda", dtype=torch.uint8)
    t._launch(t._lib.grf_bctx_gemm, t.fused, g, x.data_ptr(), x.stride(0), m, got.data_ptr(), got.stride(0), None,
              space.data_ptr(), space.numel(), t.error.data_ptr())
    assert not torch.isnan(want).any() and torch.equal(got, want)


_tensors = {}  # the last matrix: the row counts share it
