"""A predictive tensor whose matrix-core products take lookups of their own (FramePlan.for_matrix_cores)."""
import numpy as np
import pytest

from conftest import bf16_words, weight_like, words_to_float

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("walked")]


@pytest.mark.parametrize("shape", [(200, 1280), (67, 320), (530, 2048)])
def test_products_with_lookups_of_their_own(shape, monkeypatch):
    import torch
    from georefine_amd import _fused
    from georefine_amd import bitexact_predictive_codec as predictive
    from georefine_amd.bitexact_predictive_gpu import HipPredictiveGroup, HipPredictiveTensor
    rng = np.random.default_rng(shape[0])
    target = weight_like(rng, *shape)
    ref = bf16_words((target.astype(np.uint32) << 16).view(np.float32) + rng.normal(0, 0.003, shape).astype(np.float32))
    frame = predictive.encode(target, ref)
    one = HipPredictiveTensor(frame, ref)
    assert one.fused is not None and one.fused_matrix is one.fused_gemm
    monkeypatch.setattr(_fused.FramePlan, "for_matrix_cores", _fused.FramePlan.with_lookups)
    two = HipPredictiveTensor(frame, ref)
    copy = two.clone()
    assert two.fused_matrix.lognb == 10 and two.fused_gemm.lognb == 12 and two.fused.lognb == one.fused.lognb
    assert two.resident_bytes >= one.resident_bytes + two.buffers["fused_matrix_lut"].numel()
    assert copy.fused_matrix.lut not in (two.fused_matrix.lut, copy.fused_gemm.lut)
    xw = bf16_words(rng.normal(0, 1, size=(128, shape[1])))
    x = torch.from_numpy(xw).view(torch.bfloat16).cuda()
    xf, wf = words_to_float(xw).astype(np.float64), words_to_float(target).astype(np.float64)
    want, scale = xf @ wf.T, np.abs(xf) @ np.abs(wf).T
    for t in (two, copy):
        assert np.array_equal(t.decode(None).view(torch.int16).cpu().numpy().view(np.uint16), target)
        assert torch.equal(t.linear(None, x[:1], check=True), one.linear(None, x[:1]))
        for m in (2, 16, 17, 40, 96, 128):
            got = words_to_float(t.linear(None, x[:m], check=True).view(torch.uint16).cpu().numpy()).astype(np.float64)
            # one rounding to BF16, and an fp32 sum of as many terms as the matrix has columns
            assert np.all(np.abs(got - want[:m]) <= 2.0 ** -8 * np.abs(want[:m]) + shape[1] * 2.0 ** -24 * scale[:m]), m
    mixed, plain = HipPredictiveGroup([two, one, copy]), HipPredictiveGroup([one, one, one])
    for a, b in zip(mixed.linear(x[:40], check=True), plain.linear(x[:40], check=True)):
        assert torch.equal(a, b)
