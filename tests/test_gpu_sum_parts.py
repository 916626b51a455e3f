"""The parts of a product cut along K are added in their order, then the bias, and rounded once: bit for bit
what a host sum over the parts in the workspace gives, for part counts around the four read at a time."""
import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("walked")]


@pytest.mark.parametrize("parts", [2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("m", [1, 40])
def test_parts_are_added_in_order(monkeypatch, m, parts):
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    rng = np.random.default_rng(parts)
    shape = 300, 2304  # rows past one block of the sum's threads; 144 segments, 36 of four lanes
    words = (rng.choice([0x3C00, 0xBC20, 0x3D00], shape) | rng.integers(0, 32, shape)).astype(np.uint16)
    monkeypatch.setenv("GEOREFINE_FUSED_GEMM_TILING", f"4,16,{parts}")
    t = HipContextTensor(codec.encode(words), fused_segment=16)
    g = t._gemm_tiling()[0]
    assert g.k_parts == parts
    x = torch.from_numpy(rng.standard_normal((m, shape[1]), dtype=np.float32)).cuda().bfloat16()
    bias = torch.from_numpy(rng.standard_normal(shape[0], dtype=np.float32)).cuda().bfloat16()
    y = torch.empty(m, shape[0], device="cuda", dtype=torch.bfloat16)
    space = torch.empty(t._lib.grf_gemm_workspace_bytes_split(shape[1], shape[0], parts, m), device="cuda", dtype=torch.uint8)
    for b in (None, bias):
        t._launch(t._lib.grf_bctx_gemm, t.fused, g, x.data_ptr(), x.stride(0), m, y.data_ptr(), y.stride(0),
                  None if b is None else b.data_ptr(), space.data_ptr(), space.numel(), t.error.data_ptr())
        at = space.numel() - parts * m * shape[0] * 4
        shares = space[at:].view(torch.float32).reshape(parts, m, shape[0]).cpu()
        want = shares[0].clone()
        for k in range(1, parts):
            want += shares[k]
        if b is not None:
            want += b.float().cpu()
        assert torch.isfinite(want).all() and want.abs().max() > 0
        assert torch.equal(y.cpu(), want.bfloat16())
