"""Predictive matrices held as planes: the same answers as the walk's, and the walk's arrays beside them."""
import ctypes

import numpy as np
import pytest

from conftest import bf16_words, weight_like

pytestmark = pytest.mark.gpu


def _pair(rng, rows, cols):
    target = weight_like(rng, rows, cols)
    near = (target.astype(np.uint32) << 16).view(np.float32) + rng.normal(0, 0.002, (rows, cols)).astype(np.float32)
    return target, bf16_words(near)


@pytest.mark.parametrize("rows,cols", [(517, 1056), (1024, 2080)])
def test_products_decode_and_the_walks_arrays(rows, cols, monkeypatch):
    import torch
    from georefine_amd import _planes
    from georefine_amd import bitexact_predictive_codec as codec
    from georefine_amd.bitexact_context_gpu import PackedActivations
    from georefine_amd.bitexact_predictive_gpu import HipPredictiveGroup, HipPredictiveTensor
    rng = np.random.default_rng(rows)
    target, near = _pair(rng, rows, cols)
    frame = codec.encode(target, near)
    t = HipPredictiveTensor(frame, near)
    other, open_one = t.clone(), HipPredictiveTensor(frame, near, resident_contexts=False)
    assert t._planes is not None and t.has_contexts and t.fusable and open_one._planes is None
    with monkeypatch.context() as walked:
        walked.setattr(_planes, "FROM_WEIGHTS", 1 << 40)
        w = HipPredictiveTensor(frame, near)
    assert w._planes is None and t.resident_bytes <= _planes.MEMORY * w.resident_bytes
    assert [getattr(t, k) for k in ("shape", "mode", "resident_mode", "frame_bytes", "source_sha256", "reference_sha256", "frame_sha256")] == \
        [getattr(w, k) for k in ("shape", "mode", "resident_mode", "frame_bytes", "source_sha256", "reference_sha256", "frame_sha256")]
    assert np.array_equal(t.decode(None).view(torch.int16).cpu().numpy().view(np.uint16), target)
    x = torch.from_numpy(bf16_words(rng.normal(0, 1, (140, cols)))).view(torch.bfloat16).cuda()
    bias = torch.from_numpy(rng.standard_normal(rows, dtype=np.float32)).cuda().bfloat16()
    exact = x.double().cpu() @ torch.from_numpy((target.astype(np.uint32) << 16).view(np.float32)).double().T
    scale = x.double().cpu().abs() @ torch.from_numpy((target.astype(np.uint32) << 16).view(np.float32)).double().abs().T
    whole = t.gemm(None, x)
    # one rounding to BF16 and cols additions of fp32, each 2^-24 of the sum of magnitudes
    assert bool(((whole.cpu().double() - exact).abs() <= exact.abs() * 2.0 ** -8 + scale * cols * 2.0 ** -24).all())
    small = HipPredictiveTensor(codec.encode(target[:40], near[:40]), near[:40])
    group = HipPredictiveGroup([t, small, other])
    for m in (1, 7, 33, 128, 140):
        want = t.linear(None, x[:m], bias, batch_invariant=True)
        got = group.linear(x[:m], [bias, None, None], batch_invariant=True)
        assert torch.equal(got[0], want) and torch.equal(got[2], whole[:m]) and torch.equal(got[1], small.linear(None, x[:m], batch_invariant=True))
    assert torch.equal(t.linear(None, PackedActivations(x[:9])), whole[:9]) and torch.equal(t.gemv(None, x[:8]), whole[:8])
    with pytest.raises(ValueError):
        t.gemv(None, x[:9])
    # the frame's arrays, the same as of one that is walked, and what calls run is what they ran before
    for name, array in w.buffers.items():
        mine = t.buffers[name]
        assert mine.dtype == array.dtype and (name == "context_bins" or torch.equal(mine, array)), name
    assert set(t.buffers) == set(w.buffers) and t.resident_bytes > other.resident_bytes
    # (the plane of bins where it is read)
    own = torch.empty(t.shape, device="cuda", dtype=torch.int16)
    t._launch(t._lib.grf_ppcx_fused_decode, ctypes.byref(t.fused), ctypes.byref(t._tiling_for("waves")[0]), t.buffers["context_bins"].data_ptr(),
              own.data_ptr(), t.error.data_ptr())
    assert np.array_equal(own.cpu().numpy().view(np.uint16), target) and t.error.item() == 0
    assert torch.equal(t.decode(None).view(torch.int16), other.decode(None).view(torch.int16))
    assert torch.equal(t.gemm(None, x), whole) and torch.equal(group.linear(x[:20], batch_invariant=True)[0], whole[:20])
    ref = torch.from_numpy(near.view(np.int16)).view(torch.bfloat16).cuda()
    assert np.array_equal(other.decode(ref, general=True).view(torch.int16).cpu().numpy().view(np.uint16), target)
