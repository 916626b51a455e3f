"""The product of many rows with a matrix that is held as planes, against float64."""
import numpy as np
import pytest

from conftest import weight_like

pytestmark = pytest.mark.gpu


def _launch(fn, *args):
    import torch
    assert fn(*args, torch.cuda.current_stream().cuda_stream) == 0


# whole and shorter visits, units of columns that end within one, rows that end within blocks and tiles, many listed words
@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("rows,cols,parts,m,listed", [(1, 16, 1, 1, 0), (17, 240, 1, 130, 0.01), (31, 256, 1, 129, 0), (300, 1040, 1, 257, 0.01),
                                                      (513, 2320, 10, 33, 0.01), (257, 4112, 3, 300, 0.2), (784, 512, 2, 511, 0.01),
                                                      (250, 768, 3, 128, 0.9), (256, 16128, 1, 129, 0)])
def test_against_float64_and_nothing_around_is_written(tile, rows, cols, parts, m, listed):
    import torch
    from georefine_amd import _native
    from georefine_amd._planes import Planes
    lib, rng = _native.hip(), np.random.default_rng(rows + cols)
    words = weight_like(rng, rows, cols)
    words[rng.random((rows, cols)) < listed] = 0
    p = Planes.of_words(torch.from_numpy(words.view(np.int16)).cuda(), _launch)
    around = torch.full((m + 2, cols + 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    x = around[1:m + 1, :cols]
    x.copy_(torch.from_numpy(rng.standard_normal((m, cols), dtype=np.float32)))
    bias = torch.from_numpy(rng.standard_normal(rows, dtype=np.float32)).cuda().bfloat16()
    plan = parts << 16 | tile
    size = lib.grf_planes_prompt_workspace_bytes(rows, m, plan)
    assert (size > 0) == (parts > 1)
    space = torch.full((size // 4 + 64,), 5.0, device="cuda", dtype=torch.float32)
    w, xd = torch.from_numpy((words.astype(np.uint32) << 16).view(np.float32)).double(), x.cpu().double()
    ldy = rows + 3 if rows % 2 else rows  # (rows of y that begin anywhere, and on eight bytes)
    for b in (None, bias):
        y = torch.full((m + 2, ldy), 7.0, device="cuda", dtype=torch.bfloat16)
        to = y.view(-1)[(ldy + 3) // 4 * 4:]  # 8-byte aligned
        _launch(lib.grf_planes_prompt, p.address, x.data_ptr(), cols + 8, m, plan, to.data_ptr(), ldy, b.data_ptr() if b is not None else None,
                space.data_ptr(), size)
        got = to[:m * ldy].view(m, ldy)
        exact = xd @ w.T + (b.cpu().double() if b is not None else 0)
        # one rounding to BF16 (2^-9 of the value) and cols additions of fp32, each 2^-24 of the sum of magnitudes
        bound = exact.abs() * 2.0 ** -8 + (xd.abs() @ w.abs().T + 8) * cols * 2.0 ** -24
        assert bool(((got[:, :rows].cpu().double() - exact).abs() <= bound).all())
        assert bool((got[:, rows:] == 7).all() and (to[m * ldy:] == 7).all() and (y.view(-1)[:(ldy + 3) // 4 * 4] == 7).all())
        assert bool((space[size // 4:] == 5).all())


def test_linear_takes_it_where_only_values_are_asked_for_and_the_dense_way_elsewhere():
    import torch
    from georefine_amd import _native
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    rng, rows, cols, m = np.random.default_rng(2), 3000, 4096, 150
    assert _native.hip().grf_planes_prompt_plan(rows, cols, m) >= 0
    words = weight_like(rng, rows, cols)
    tensor = HipContextTensor(codec.encode(words), device="cuda:0")
    x = torch.from_numpy(rng.standard_normal((3, m // 3, cols), dtype=np.float32)).cuda().bfloat16()
    w = torch.from_numpy(words.view(np.int16)).cuda().view(torch.bfloat16)
    want = x.double() @ w.double().T
    bound = want.abs() * 2.0 ** -8 + x.double().abs() @ w.double().abs().T * cols * 2.0 ** -24
    wide = torch.zeros(m, cols + 8, device="cuda", dtype=torch.bfloat16)
    wide[:, :cols] = x.view(m, cols)
    for given in (x, wide[:, :cols].view(3, m // 3, cols), x.transpose(1, 2).contiguous().transpose(1, 2), x[:1].expand(3, -1, -1)):
        exact, near = (want, bound) if given.stride(0) else (want[:1].expand(3, -1, -1), bound[:1].expand(3, -1, -1))
        assert bool(((tensor.linear(given).double() - exact).abs() <= near).all())
    asked = x.clone().requires_grad_()
    y = tensor.linear(asked)
    y.backward(torch.ones_like(y))
    assert bool(((y.detach().double() - want).abs() <= bound).all())
    assert torch.allclose(asked.grad.double(), w.double().sum(0).expand_as(x), rtol=2.0 ** -7, atol=2.0 ** -7)
    with pytest.raises(RuntimeError):
        tensor.linear(x[..., :-16])
    with pytest.raises(RuntimeError):
        tensor.linear(x.float())
