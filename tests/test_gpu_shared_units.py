"""More than 64 rows on matrix-core launches whose workgroups share compute units: the same bits a row has in a smaller batch."""
import numpy as np
import pytest

from georefine_amd import bitexact_context_codec as codec

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("walked")]


@pytest.mark.parametrize("rows,cols,members", [(2048, 5120, 1), (2047, 5104, 1), (4096, 2560, 2), (1024, 5120, 1)])
def test_rows_keep_their_bits_above_64(rows, cols, members):
    import torch
    from georefine_amd.bitexact_context_gpu import HipContextTensor, HipLinearGroup
    rng = np.random.default_rng(cols)
    ws = [torch.from_numpy((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)).bfloat16() for _ in range(members)]
    ts = [HipContextTensor(codec.encode(w.view(torch.int16).numpy().view(np.uint16)), residual_block=16) for w in ws]
    call = (lambda v: HipLinearGroup(ts).linear(v, batch_invariant=True)) if members > 1 else (
        lambda v: [ts[0].linear(v, batch_invariant=True)])
    x = torch.from_numpy(rng.standard_normal((128, cols)).astype(np.float32)).bfloat16().cuda()
    x[70] = float("inf")
    parts = [torch.cat(halves) for halves in zip(call(x[:64]), call(x[64:].contiguous()))]
    for m in (65, 80, 96, 97, 128):
        for got, expect in zip(call(x[:m].contiguous()), parts):
            assert torch.equal(got.view(torch.int16), expect[:m].view(torch.int16)), m
    exact = x[:64].cpu().double() @ ws[0].double().T
    bound = exact.abs() * 2.0 ** -8 + (x[:64].cpu().double().abs() @ ws[0].double().abs().T) * cols * 2.0 ** -24
    assert bool(((parts[0][:64].double().cpu() - exact).abs() <= bound).all())
