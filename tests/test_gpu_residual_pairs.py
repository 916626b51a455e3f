"""Residual groups in pair form: what a group's bits become, and both forms through every kernel."""
import copy
import ctypes

import numpy as np
import pytest

from tests.conftest import bf16_words, weight_like

pytestmark = pytest.mark.gpu


def _pair_form(packed):
    """The rule of the header in numpy: 12-byte groups of sixteen 6-bit fields, most significant bit first."""
    bits = np.unpackbits(packed.reshape(-1, 12), axis=1).reshape(-1, 16, 6)
    fields = (bits * (32, 16, 8, 4, 2, 1)).sum(2).astype(np.uint64)
    word = (fields & np.uint64(31)) | (fields >> np.uint64(5)) << np.uint64(15)
    p = [word[:, 2 * i] | word[:, 2 * i + 1] << np.uint64(16) for i in range(8)]
    rol = lambda v, by: (v << np.uint64(by) | v >> np.uint64(32 - by)) & np.uint64(0xFFFFFFFF)
    inner, outer = np.uint64(0x001E001E), np.uint64(0x80018001)
    dwords = (p[0] | rol(p[1], 6) | rol(p[6] & inner, 10), p[2] | rol(p[3], 6) | rol(p[7] & inner, 10),
              p[4] | rol(p[5], 6) | rol(p[6] & outer, 12) | rol(p[7] & outer, 14))
    return np.stack(dwords, 1).astype(np.uint32).view(np.uint8).reshape(-1)


@pytest.mark.parametrize("groups", [1, 2, 255, 257, 70001])
def test_pair_form_and_back(groups):
    import torch
    from georefine_amd.bitexact_context_gpu import _residual_form
    packed = np.random.default_rng(groups).integers(0, 256, 12 * groups, dtype=np.uint8)
    if groups == 2:
        packed[:] = (0xFF,) * 12 + (0,) * 12
    on_device = torch.from_numpy(packed).cuda()
    _residual_form(on_device, True)
    assert np.array_equal(on_device.cpu().numpy(), _pair_form(packed))
    assert np.array_equal(_residual_form(on_device, False).cpu().numpy(), packed)


def test_groups_are_checked():
    import torch
    from georefine_amd import _native
    lib, data = _native.hip(), torch.zeros(64, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.grf_pair_residuals(data.data_ptr(), 24, 1, stream) == 0 and lib.grf_pair_residuals(data.data_ptr(), 0, 1, stream) == 0
    for args in ((None, 24), (data.data_ptr() + 2, 24), (data.data_ptr(), 25)):
        assert lib.grf_pair_residuals(*args, 1, stream) != 0 and b"grf_pair_residuals" in lib.grf_last_error()
    torch.cuda.synchronize()


@pytest.mark.parametrize("segment", [16, 32, 64])
def test_both_forms_give_the_same_words_and_products(segment):
    import torch
    from georefine_amd import _hip_abi
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor, HipLinearGroup
    words = weight_like(np.random.default_rng(segment), 150, 1024)
    pairs = HipContextTensor(codec.encode(words), device="cuda:0", fused_segment=segment)
    assert pairs.fused.nc & _hip_abi.RAW_PAIRS and "residual_stream" not in pairs.buffers
    fields = copy.copy(pairs)
    fields.buffers = dict(pairs.buffers)
    fields.buffers["residual_stream"] = pairs.buffers["residual_stream"]
    fields._bind()
    assert not fields.fused.nc & _hip_abi.RAW_PAIRS
    ids = torch.tensor([149, 0, 7, 7], device="cuda")
    for t in (pairs, fields):
        for got in (t.decode(), t.decode(general=True)):
            assert np.array_equal(got.view(torch.uint16).cpu().numpy(), words)
        assert np.array_equal(t.gather_rows(ids).view(torch.uint16).cpu().numpy(), words[ids.cpu().numpy()])
    for m in (1, 2, 5, 20, 40, 100):
        x = torch.from_numpy(bf16_words(np.random.default_rng(m).normal(0, 1, (m, 1024)))).view(torch.bfloat16).cuda()
        want = pairs.gemm(x, check=True)
        assert torch.equal(fields.gemm(x, check=True), want)
        if m <= 8:
            assert torch.equal(fields.gemv(x, check=True), pairs.gemv(x, check=True))
        group = lambda t: HipLinearGroup([t, t]).linear(x, check=True)
        assert all(torch.equal(a, b) for a, b in zip(group(fields), group(pairs)))
    with pytest.raises(codec.CodecError, match="one form"):
        HipLinearGroup([pairs, fields]).linear(x)
    flagged = type(pairs._frame).from_buffer_copy(pairs._frame)
    flagged.mode = 128  # (a rANS residual stream has no pair form)
    out = torch.empty(words.size, dtype=torch.uint16, device="cuda")
    assert pairs._lib.grf_bctx_decode(ctypes.byref(flagged), None, 1, out.data_ptr(), pairs.error.data_ptr(),
                                      torch.cuda.current_stream().cuda_stream) != 0
