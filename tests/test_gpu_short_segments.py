"""Products, decode and lookups of matrices indexed at sixteen-symbol segments, the length the smallest ones get."""
import numpy as np
import pytest

from georefine_amd import bitexact_context_codec as codec

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("walked")]


@pytest.mark.parametrize("rows,cols", [(256, 512), (257, 560), (1000, 1040), (3839, 1024), (900, 4096)])
def test_smallest_matrices_against_their_words(rows, cols):
    import torch
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    rng = np.random.default_rng(rows)
    w = torch.from_numpy((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)).bfloat16()
    words = w.view(torch.int16).numpy().view(np.uint16)
    t = HipContextTensor(codec.encode(words))
    assert t.fused is not None and t.fused_plan["seg_len"] == 16
    assert torch.equal(t.decode().cpu().view(torch.int16), w.view(torch.int16))
    ids = torch.from_numpy(rng.integers(0, rows, 33)).cuda()
    assert torch.equal(t.gather_rows(ids).cpu().view(torch.int16), w[ids.cpu()].view(torch.int16))
    for m in (1, 2, 3, 16, 17, 64, 65, 128):
        x = torch.from_numpy(rng.standard_normal((m, cols)).astype(np.float32)).bfloat16()
        got = t.linear(x.cuda()).double().cpu()
        exact = x.double() @ w.double().T
        # one rounding to BF16 (2^-9 of the value) and cols fp32 additions of products, each 2^-24 of the sum of magnitudes
        bound = exact.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().T) * cols * 2.0 ** -24
        assert bool(((got - exact).abs() <= bound).all()), m
