"""Small products on the matrix cores read the activations where they are: the same bits as from
the packed copy, and nothing of what lies around the rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols,segment", [(64 * 5, 64), (16 * 9, 16), (64 * 33, 64)])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 33, 64, 65])
def test_rows_in_place_equal_the_packed_copy(m, cols, segment):
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor, HipLinearGroup, PackedActivations
    rng = np.random.default_rng(cols + m)
    ts = [HipContextTensor(codec.encode((rng.choice([0x3C00, 0x3C20, 0x3D00], (rows, cols))
                                         | rng.integers(0, 32, (rows, cols))).astype(np.uint16)), fused_segment=segment)
          for rows in (83, 160)]
    for pad, first in ((0, 0), (8, 0), (4, 4)):  # contiguous; rows apart; rows on 8-byte boundaries
        around = torch.full((m + 2, cols + pad), float("nan"), device="cuda", dtype=torch.bfloat16)
        x = around.view(-1)[first:first + (m + 1) * (cols + pad)].view(m + 1, cols + pad)[1:, :cols]
        x.copy_(torch.from_numpy(rng.standard_normal((m, cols), dtype=np.float32)))
        expected = [t.gemm(PackedActivations(x)) for t in ts]
        assert not any(torch.isnan(y).any() for y in expected)
        for t, y in zip(ts, expected):
            got = torch.empty_like(y)
            space = torch.empty(1 << 20, device="cuda", dtype=torch.uint8)
            tiling = t._gemm_tiling()[0]
            t._launch(t._lib.grf_bctx_gemm, t.fused, tiling, x.data_ptr(), x.stride(0), m, got.data_ptr(), got.stride(0),
                      None, space.data_ptr(), space.numel(), t.error.data_ptr())
            assert torch.equal(got, y)
        grouped = HipLinearGroup(ts).linear(x, batch_invariant=True)
        packed = HipLinearGroup(ts).linear(PackedActivations(x))
        assert all(torch.equal(a, b) for a, b in zip(grouped, packed))
