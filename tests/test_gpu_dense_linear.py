"""Products of more rows than the fused kernels take: the matrix-core kernel over the decoded matrix."""
import ctypes

import numpy as np
import pytest

from tests.conftest import bf16_words, weight_like

pytestmark = pytest.mark.gpu


def _reference(x, w, bias):
    """(float64 product, what BF16 and fp32 sums may be off by): one rounding of the result, 2^-9 of it, and as
    many fp32 roundings of the running sum as there are terms, 2^-24 each of at most the sum of magnitudes."""
    want = x.double() @ w.double().T
    scale = x.double().abs() @ w.double().abs().T
    if bias is not None:
        want, scale = want + bias.double(), scale + bias.double().abs()
    return want, want.abs() * 2.0 ** -8 + scale * (w.shape[1] + 64) * 2.0 ** -24


def _product(x, w, bias):
    import torch
    from georefine_amd import _native
    lib = _native.hip()
    (m, cols), rows = x.shape, w.shape[0]
    y = torch.full((m, rows), float("nan"), device="cuda", dtype=torch.bfloat16)
    size = lib.grf_dense_gemm_workspace_bytes(rows, cols, m)
    space = torch.empty(size // 4 + 4, device="cuda", dtype=torch.float32).fill_(float("nan"))
    assert lib.grf_dense_gemm(w.data_ptr(), rows, cols, x.data_ptr(), x.stride(0), m, y.data_ptr(), rows,
                              bias.data_ptr() if bias is not None else None, space.data_ptr(), size,
                              torch.cuda.current_stream().cuda_stream) == 0, lib.grf_last_error()
    return y, size


# rows x cols at m rows: each tile (256 x 256, 256 x 192, 256 x 128, 128 x 128, 128 x 64), cut along K and whole, with rows
# and columns that do and do not end on a tile, on a step of 64 columns, on four rows; fewer columns than a step, than two;
# one row and column
SHAPES = [(1, 1, 8), (129, 65, 24), (130, 63, 64), (128, 64, 128), (257, 127, 72), (129, 300, 136), (200, 255, 528), (256, 256, 2048),
          (257, 770, 16), (300, 4099, 1040), (1000, 2050, 600), (513, 2305, 10304), (1000, 1028, 16448), (160, 5120, 17408),
          (129, 257, 1032), (257, 2049, 1032), (257, 2049, 4104), (129, 4100, 4104), (257, 12290, 1032), (1000, 3001, 4104),
          (1000, 8193, 520), (129, 12290, 4104), (1000, 12290, 1032)]


@pytest.mark.parametrize("m,rows,cols", SHAPES)
def test_product_at_the_edges_of_tiles(m, rows, cols):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(m * 31 + rows * 7 + cols)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=g).bfloat16()
    wide = torch.full((m, cols + 24), float("nan"), device="cuda", dtype=torch.bfloat16)  # rows further apart than they are long
    wide[:, :cols] = draw(m, cols)
    x, w, bias = wide[:, :cols], draw(rows, cols), draw(rows)
    want, off = _reference(x, w, bias)
    y, _ = _product(x, w, bias)
    assert bool(((y.double() - want).abs() <= off).all())
    assert torch.equal(_product(x, w, bias)[0], y)  # a fixed order of additions
    want, off = _reference(x, w, None)
    assert bool(((_product(x.contiguous(), w, None)[0].double() - want).abs() <= off).all())


def test_linear_takes_it_and_leaves_the_rest_to_torch():
    import torch
    from georefine_amd import _native
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    words = weight_like(np.random.default_rng(5), 640, 512)
    t = HipContextTensor(codec.encode(words), device="cuda:0")
    dense = t.decode()
    assert _native.hip().grf_dense_gemm_plan(640, 512, 150) >= 0
    x = torch.from_numpy(bf16_words(np.random.default_rng(6).normal(0, 1, (150, 512)))).view(torch.bfloat16).cuda()
    bias = torch.from_numpy(bf16_words(np.random.default_rng(7).normal(0, 1, 640))).view(torch.bfloat16).cuda()
    want, off = _reference(x, dense, bias)
    near = lambda y: bool(((y.detach().double().reshape(want.shape) - want).abs() <= off).all())
    own = t.linear(x, bias, check=True)
    assert near(own) and torch.equal(own, _product(x, dense, bias)[0])
    for form in (x.view(3, 50, 512), x.t().contiguous().t(), torch.cat((x, x), 1)[:, :512], x.reshape(-1)[None].view(150, 512),
                 torch.cat((x.new_zeros(1), x.reshape(-1)))[1:].view(150, 512)):  # shapes, orders, strides, alignment
        y = t.linear(form, bias)
        assert y.shape == (*form.shape[:-1], 640) and near(y)
    one = x[:1].expand(150, 512)  # rows that are one row
    assert torch.equal(t.linear(one, bias), t.linear(one.contiguous(), bias))
    leaf = x.clone().requires_grad_()
    y = t.linear(leaf, bias)
    assert near(y) and y.requires_grad
    y.sum().backward()
    assert leaf.grad.shape == x.shape
    with torch.autograd.forward_ad.dual_level():  # (linear: the tangent along x is the value)
        value, tangent = torch.autograd.forward_ad.unpack_dual(t.linear(torch.autograd.forward_ad.make_dual(x, x)))
        assert torch.equal(value, tangent)
    with pytest.raises(RuntimeError):
        t.linear(x.float(), bias)
    with pytest.raises(RuntimeError):
        t.linear(x, bias[:-1])
    with pytest.raises(RuntimeError):
        t.linear(x[:, :256], bias)


def test_arguments_are_checked_before_anything_is_launched():
    import torch
    from georefine_amd import _native
    lib = _native.hip()
    x, w, y = (torch.zeros(256, 1024, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    good = dict(w=w.data_ptr(), rows=200, cols=1024, x=x.data_ptr(), ldx=1024, m=200, y=y.data_ptr(), ldy=200, bias=None,
                space=None, size=0)
    call = lambda **k: lib.grf_dense_gemm(*{**good, **k}.values(), torch.cuda.current_stream().cuda_stream)
    need = lib.grf_dense_gemm_workspace_bytes(200, 1024, 200)
    space = torch.empty(need // 4 + 4, device="cuda", dtype=torch.float32)
    assert need and call(space=space.data_ptr(), size=need) == 0
    for bad in (dict(), dict(space=space.data_ptr(), size=need - 1), dict(space=space.data_ptr() + 4, size=need), dict(x=None),
                dict(cols=1020), dict(ldx=1020), dict(ldx=1016), dict(ldy=199), dict(x=x.data_ptr() + 2), dict(y=y.data_ptr() + 2),
                dict(rows=0), dict(m=0)):
        assert call(**{**dict(space=space.data_ptr(), size=need), **bad} if bad else {}) != 0, bad
        assert b"grf_dense_gemm" in lib.grf_last_error()
    torch.cuda.synchronize()


def test_graph_replays_give_the_same_bits():
    import torch
    from georefine_amd import _native
    from georefine_amd.bitexact_context_gpu import dense_linear
    lib = _native.hip()
    w, x = (torch.randn(n, 1024, device="cuda").bfloat16() for n in (1024, 200))
    eager = dense_linear(lib, x, w, None, 0)
    held = x.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = dense_linear(lib, held, w, None, 0)
    for k in range(3):
        held.copy_(x * (k + 1))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, dense_linear(lib, x * (k + 1), w, None, 0)), k
    assert torch.equal(eager, dense_linear(lib, x, w, None, 0))
