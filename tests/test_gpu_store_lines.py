"""The store sink that holds words back: segments of whole lines, of half lines and of neither, whatever
the workgroup, equal the one-lane-per-segment decode, with nothing written around the matrix."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,segment", [(1, 64 * 9, 64), (37, 64 * 33, 64), (300, 128 * 5, 128), (33, 96 * 7, 96),
                                               (70, 32 * 65, 32), (41, 48 * 5, 48), (50, 16 * 3, 16)])
@pytest.mark.parametrize("forced", [None, "1024,16,8", "512,8,16", "768,32,4"])
def test_words_held_back_equal_the_general_decode(monkeypatch, forced, rows, cols, segment):
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    rng = np.random.default_rng(rows)
    words = (rng.choice([0x3C00, 0x3C20, 0xBD00], (rows, cols)) | rng.integers(0, 32, (rows, cols))).astype(np.uint16)
    if forced:
        monkeypatch.setenv("GEOREFINE_FUSED_WAVE_TILING", forced)
    t = HipContextTensor(codec.encode(words, residual="raw6"), fused_segment=segment)
    assert t.fused is not None and t.fused_plan["seg_len"] == segment
    around = torch.full((rows * cols + 256,), 0x7FC1, device="cuda", dtype=torch.int32).to(torch.uint16)
    t._launch(t._lib.grf_bctx_fused_decode, t.fused, t._store_tiling()[0], around.data_ptr() + 256, t.error.data_ptr())
    got = around.cpu().numpy()
    assert int(t.error.item()) == 0
    assert np.array_equal(got[128:-128].reshape(rows, cols), words)
    assert np.all(got[:128] == 0x7FC1) and np.all(got[-128:] == 0x7FC1)
    assert np.array_equal(t.decode(check=True, general=True).view(torch.uint16).cpu().numpy(), words)
