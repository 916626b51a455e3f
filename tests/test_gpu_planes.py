"""Matrices held as planes: every sink against the words they were laid out from."""
import numpy as np
import pytest

from conftest import bf16_words, weight_like

pytestmark = pytest.mark.gpu


def _launch(fn, *args):
    import torch
    assert fn(*args, torch.cuda.current_stream().cuda_stream) == 0


def _planes(words):
    import torch
    from georefine_amd._planes import Planes
    return Planes.of_words(torch.from_numpy(words.view(np.int16)).cuda(), _launch)


def _words(kind, rows, cols, seed):
    rng = np.random.default_rng(seed)
    if kind == "any":  # every bit pattern: most words are listed
        return rng.integers(0, 1 << 16, (rows, cols)).astype(np.uint16)
    words = weight_like(rng, rows, cols)
    words[rng.random((rows, cols)) < 0.01] = 0
    words.flat[rng.integers(0, words.size, 6)] = (0x7F80, 0xFF80, 0x7FC1, 0x0001, 0x8000, 0x7F7F)
    return words


SHAPES = [(1, 16), (16, 64), (15, 256), (17, 240), (33, 272), (16, 448), (100, 4096), (31, 4112), (257, 1040), (40, 17408)]


@pytest.mark.parametrize("kind", ["weights", "any"])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_words_and_rows_come_back_and_nothing_around_them_is_written(rows, cols, kind):
    import torch
    from georefine_amd import _native
    lib, words = _native.hip(), _words(kind, rows, cols, rows + cols)
    p = _planes(words)
    around = torch.full((rows * cols + 256,), 0x5A5A, device="cuda", dtype=torch.int16)
    _launch(lib.grf_planes_decode, p.address, around.data_ptr() + 256)
    got = around.cpu().numpy().view(np.uint16)
    assert np.array_equal(got[128:-128].reshape(rows, cols), words)
    assert np.all(got[:128] == 0x5A5A) and np.all(got[-128:] == 0x5A5A)
    ids = torch.from_numpy(np.random.default_rng(1).integers(0, rows, 19)).cuda()
    out = torch.full((21, cols), 0x5A5A, device="cuda", dtype=torch.int16)
    _launch(lib.grf_planes_gather, p.address, ids.data_ptr(), 19, out[1:].data_ptr(), None, None, None)
    got = out.cpu().numpy().view(np.uint16)
    assert np.array_equal(got[1:-1], words[ids.cpu().numpy()]) and np.all(got[0] == 0x5A5A) and np.all(got[-1] == 0x5A5A)


@pytest.mark.parametrize("splits", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_products_against_float64_with_one_set_of_bits_a_row(rows, cols, splits):
    import torch
    from georefine_amd import _hip_abi, _native
    from georefine_amd._planes import visits
    from georefine_amd.bitexact_context_gpu import PackedActivations
    if not (splits - 1) * -(-visits(cols) // splits) < visits(cols) <= 63 * splits:
        pytest.skip("splits of 1 to 63 visits")
    lib, rng = _native.hip(), np.random.default_rng(rows)
    words = weight_like(rng, rows, cols)
    words[rng.random((rows, cols)) < 0.02] = 0  # (listed)
    p = _planes(words)
    p.struct.splits = splits
    around = torch.full((130, cols + 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    x = around[1:129, :cols]  # rows apart, with what must not be read around them
    x.copy_(torch.from_numpy(rng.standard_normal((128, cols), dtype=np.float32)))
    bias = torch.from_numpy(rng.standard_normal(rows, dtype=np.float32)).cuda().bfloat16()
    space = torch.empty(splits * 128 * rows + 64, device="cuda", dtype=torch.float32)

    def product(rows_of_x, m, packed=0, b=None):
        y = torch.full((m + 2, rows), 7.0, device="cuda", dtype=torch.bfloat16)
        _launch(lib.grf_planes_linear, p.address, rows_of_x.data_ptr(), cols + 8, m, packed, y[1:].data_ptr(),
                b.data_ptr() if b is not None else None, space.data_ptr(), space.numel() * 4)
        assert bool((y[0] == 7).all() and (y[-1] == 7).all())
        return y[1:-1]

    full, shifted = product(x, 128), product(x, 128, b=bias)
    w, xd = torch.from_numpy((words.astype(np.uint32) << 16).view(np.float32)).double(), x.cpu().double()
    for got, exact in ((full, xd @ w.T), (shifted, xd @ w.T + bias.cpu().double())):
        # one rounding to BF16 (2^-9 of the value) and cols additions of fp32, each 2^-24 of the sum of magnitudes
        bound = exact.abs() * 2.0 ** -8 + (xd.abs() @ w.abs().T + 8) * cols * 2.0 ** -24
        assert bool(((got.cpu().double() - exact).abs() <= bound).all())
    for m in (1, 15, 16, 17, 32, 33, 64, 65, 127):
        assert torch.equal(product(x, m), full[:m]), m
        xp = PackedActivations(x[:m])
        assert torch.equal(product(xp.buffer, m, packed=1), full[:m]), m


# (the last: blocks that are more than units, of waves that fill one: more than sixteen rows share x)
@pytest.mark.parametrize("rows,cols", [(29968, 2320), (65555, 1040), (4112, 3328)])
def test_rows_of_x_that_large_matrices_share_have_the_bits_of_single_ones(rows, cols):
    import torch
    from georefine_amd import _native
    from georefine_amd.bitexact_context_gpu import PackedActivations
    lib, g = _native.hip(), torch.Generator(device="cuda").manual_seed(rows)
    words = (torch.randn(rows, cols, device="cuda", generator=g) * 0.02).bfloat16()
    x = torch.randn(32, cols, device="cuda", generator=g).bfloat16()
    p = _planes(words.view(torch.int16).cpu().numpy().view(np.uint16))

    def product(rows_of_x, m, packed=0):
        space = torch.empty(p.workspace(m) // 4 + 4, device="cuda", dtype=torch.float32)
        y = torch.empty(m, rows, device="cuda", dtype=torch.bfloat16)
        _launch(lib.grf_planes_linear, p.address, rows_of_x.data_ptr(), cols, m, packed, y.data_ptr(), None, space.data_ptr(), p.workspace(m))
        return y

    want = torch.cat([product(x[i:i + 1], 1) for i in range(32)])
    exact = x.double() @ words.double().T
    bound = exact.abs() * 2.0 ** -8 + x.double().abs() @ words.double().abs().T * cols * 2.0 ** -24
    assert bool(((want.double() - exact).abs() <= bound).all())
    for m in (8, 9, 16, 17, 32):
        assert torch.equal(product(x, m), want[:m]), m
        assert torch.equal(product(PackedActivations(x[:m]).buffer, m, packed=1), want[:m]), m


@pytest.mark.parametrize("rows,cols,splits", [(4097, 17408, 12), (4200, 16400, 13)])
def test_row_blocks_that_workgroups_share_give_the_bits_of_whole_ones(rows, cols, splits):
    import torch
    from georefine_amd import _native
    lib, g = _native.hip(), torch.Generator(device="cuda").manual_seed(rows)
    words = (torch.randn(rows, cols, device="cuda", generator=g) * 0.02).bfloat16()
    words.view(-1)[torch.randint(0, rows * cols, (100000,), device="cuda", generator=g)] = 0  # (listed)
    x = torch.randn(8, cols, device="cuda", generator=g).bfloat16()
    bias = torch.randn(rows, device="cuda", generator=g).bfloat16()
    from georefine_amd._planes import Planes
    p = Planes.of_words(words.view(torch.int16), _launch)
    p.struct.splits = splits
    size = p.workspace(8)
    assert size >= splits * 8 * rows * 4
    space = torch.full((size // 4 + 64,), 5.0, device="cuda", dtype=torch.float32)
    exact = x.double() @ words.double().T + bias.double()
    bound = exact.abs() * 2.0 ** -8 + (x.double().abs() @ words.double().abs().T + 8) * cols * 2.0 ** -24
    for m in (1, 2, 7, 8):
        whole, absent, askew, shared = (torch.full((m + 2, rows), 7.0, device="cuda", dtype=torch.bfloat16) for _ in range(4))
        # without a workspace blocks are whole, and one that is null or not aligned is none
        for y, s, n in ((whole, None, 0), (absent, None, size), (askew, space.data_ptr() + 4, size), (shared, space.data_ptr(), size)):
            if y is shared:
                assert bool((space == 5).all())
            _launch(lib.grf_planes_linear, p.address, x.data_ptr(), cols, m, 0, y[1:].data_ptr(), bias.data_ptr(), s, n)
        assert torch.equal(whole, shared) and bool((shared[0] == 7).all() and (shared[-1] == 7).all())
        assert torch.equal(whole, absent) and torch.equal(whole, askew) and bool((space[size // 4:] == 5).all())
        space.fill_(5)
        assert bool(((shared[1:-1].double() - exact[:m]).abs() <= bound[:m]).all())


def test_members_of_more_splits_than_the_largest_one_have_two_a_wave():
    import ctypes
    import torch
    from georefine_amd import _native
    lib, rng, cols = _native.hip(), np.random.default_rng(9), 2320  # ten visits
    members = [_planes(weight_like(rng, rows, cols)) for rows in (900, 70, 33)]
    for p, splits in zip(members, (3, 5, 10)):  # (the last one's ten need waves of two where three would do)
        p.struct.splits = splits
    x = torch.from_numpy(rng.standard_normal((40, cols), dtype=np.float32)).cuda().bfloat16()
    for m in (1, 8, 12, 31, 40):
        space = torch.empty(1 << 20, device="cuda", dtype=torch.float32)
        alone, together = ([torch.empty(m, p.rows, device="cuda", dtype=torch.bfloat16) for p in members] for _ in range(2))
        for p, y in zip(members, alone):
            _launch(lib.grf_planes_linear, p.address, x.data_ptr(), cols, m, 0, y.data_ptr(), None, space.data_ptr(), space.numel() * 4)
        for order in ((0, 1, 2), (2, 1, 0), (1, 2)):
            n, of = len(order), lambda kind, values: (kind * len(values))(*values)
            _launch(lib.grf_planes_group, n, of(ctypes.c_void_p, [members[i].address for i in order]), x.data_ptr(), cols, m, 0,
                    of(ctypes.c_void_p, [together[i].data_ptr() for i in order]), of(ctypes.c_uint32, [members[i].rows for i in order]), None,
                    space.data_ptr(), space.numel() * 4)
            assert all(torch.equal(together[i], alone[i]) for i in order), (m, order)


@pytest.mark.parametrize("splits", [11, 14, 15, 16])
def test_rows_past_eight_of_many_splits_fit_in_a_units_memory(splits):
    import torch
    from georefine_amd import _native
    from georefine_amd.bitexact_context_gpu import PackedActivations
    lib, rng, rows, cols = _native.hip(), np.random.default_rng(splits), 50, splits * 256 - 80
    p = _planes(weight_like(rng, rows, cols))
    p.struct.splits = splits
    x = torch.from_numpy(rng.standard_normal((33, cols), dtype=np.float32)).cuda().bfloat16()
    space = torch.empty(splits * 64 * rows, device="cuda", dtype=torch.float32)

    def product(rows_of_x, m, packed=0):
        y = torch.empty(m, rows, device="cuda", dtype=torch.bfloat16)
        _launch(lib.grf_planes_linear, p.address, rows_of_x.data_ptr(), cols, m, packed, y.data_ptr(), None, space.data_ptr(), space.numel() * 4)
        return y

    want = product(x, 33)
    for m in (1, 8, 9, 16, 17, 32):
        assert torch.equal(product(x, m), want[:m]), m
        assert torch.equal(product(PackedActivations(x[:m]).buffer, m, packed=1), want[:m]), m


def test_infinities_and_nan_go_where_the_dense_product_puts_them():
    import torch
    from georefine_amd import _native
    rng = np.random.default_rng(8)
    words = weight_like(rng, 40, 544) & 0x7FFF  # positive: an infinite activation gives no NaN
    words[3, 500], words[5, 7], words[6, 100], words[7, :] = 0x7F80, 0x7FC0, 0, 0x3F80
    p = _planes(words)
    dense = torch.from_numpy(words.view(np.int16)).view(torch.bfloat16).cuda()
    space = torch.empty(1 << 16, device="cuda", dtype=torch.float32)
    for m in (1, 20, 64, 70):
        x = torch.from_numpy(rng.random((m, 544), dtype=np.float32) + 0.5).cuda().bfloat16()
        x[0, 100] = float("inf")
        x[m - 1, 543] = float("nan") if m > 1 else x[0, 543]
        y = torch.empty(m, 40, device="cuda", dtype=torch.bfloat16)
        _launch(_native.hip().grf_planes_linear, p.address, x.data_ptr(), 544, m, 0, y.data_ptr(), None, space.data_ptr(), space.numel() * 4)
        want = x.double() @ dense.double().T
        for state in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(state(y), state(want)), (m, state)


def test_a_tensor_answers_as_planes_whatever_is_looked_at():
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor, HipLinearGroup
    rng = np.random.default_rng(12)
    words = weight_like(rng, 700, 1040)
    for residual in ("auto", "raw6"):
        frame = codec.encode(words, residual=residual)
        t = HipContextTensor(frame)
        assert t.fusable and t._planes is not None and t.fused_reason == ""
        other, small = t.clone(residual_block=16), HipContextTensor(codec.encode(weight_like(rng, 48, 1040)))
        assert small._planes is None
        held = small.resident_bytes
        group, alone = HipLinearGroup([t, small, other]), HipLinearGroup([small])
        assert small._planes is None and small.resident_bytes == held
        x = torch.from_numpy(bf16_words(rng.normal(0, 1, (140, 1040)))).view(torch.bfloat16).cuda()
        for m in (1, 2, 20, 128, 140):
            want = t.linear(x[:m], batch_invariant=True)
            assert torch.equal(t.linear(x[:m], batch_invariant=True, check=True), want)
            got = group.linear(x[:m], batch_invariant=True)
            assert torch.equal(got[0], want) and torch.equal(got[2], want)
            assert torch.equal(got[1], alone.linear(x[:m], batch_invariant=True)[0])
        assert torch.equal(group.linear(x[:1])[1], small.linear(x[:1]))  # (the vector-ALU route gives every member its own bits)
        ids = torch.tensor([[0, 699], [5, 5]])
        assert np.array_equal(t.gather_rows(ids).view(torch.int16).cpu().numpy().view(np.uint16), words[ids.numpy()])
        for bad in (-1, 700):
            with pytest.raises(IndexError):
                t.gather_rows(torch.tensor([3, bad]))
            last = t.gather_rows(torch.tensor([3, bad]), check=False, validate=False)[1]
            assert np.array_equal(last.view(torch.int16).cpu().numpy().view(np.uint16), words[0 if bad < 0 else 699])
        as_planes, before, grouped = t.resident_bytes, t.linear(x[:20]), group.linear(x[:20])
        assert other.resident_bytes == as_planes
        streams = HipContextTensor.host_prepare(frame)["indexed"]
        assert t.fused is not None  # the frame's arrays, the same as of one that is walked
        for name in ("main_stream", "rows", "columns", "main_freq", "fused_seg_state", "fused_seg_offset", "residual_stream"):
            assert np.array_equal(t.buffers[name].cpu().numpy()[:streams[name].size], streams[name]), name
        assert t.mode == frame[5] and t.frame_bytes == len(frame) and t.resident_bytes > as_planes == other.resident_bytes
        for general in (False, True):
            assert np.array_equal(t.decode(general=general).view(torch.int16).cpu().numpy().view(np.uint16), words)
        # and what calls run is what they ran before
        assert torch.equal(t.linear(x[:20]), before) and all(torch.equal(a, b) for a, b in zip(group.linear(x[:20]), grouped))
        assert torch.equal(grouped[0], before) and torch.equal(grouped[1], alone.linear(x[:20])[0]) and torch.equal(grouped[2], other.linear(x[:20]))
        assert np.array_equal(other.decode(general=True).view(torch.int16).cpu().numpy().view(np.uint16), words) and other._raw6_block == 16


def test_captured_launches_replay_on_new_rows():
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor, HipLinearGroup
    rng = np.random.default_rng(13)
    t = HipContextTensor(codec.encode(weight_like(rng, 640, 1024)))
    group = HipLinearGroup([t, t.clone()])
    draw = lambda m: torch.from_numpy(bf16_words(rng.normal(0, 1, (m, 1024)))).view(torch.bfloat16).cuda()
    x1, x40, ids = draw(1), draw(40), torch.from_numpy(rng.integers(0, 640, 33)).cuda()
    step = lambda: [t.linear(x1), *group.linear(x40), t.decode(check=False), t.gather_rows(ids, check=False, validate=False)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for _ in range(3):
        x1.copy_(draw(1)), x40.copy_(draw(40)), ids.copy_(torch.from_numpy(rng.integers(0, 640, 33)))
        eager = [v.clone() for v in step()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(captured, eager))
    assert t.buffers["main_stream"].is_cuda and t.decode(general=True).is_cuda
    torch.cuda.empty_cache()
    x1.copy_(draw(1)), x40.copy_(draw(40))
    graph.replay()
    want = t.linear(x1)
    assert torch.equal(captured[0], want) and torch.equal(captured[1], captured[2])


def test_captured_launches_of_a_small_member_outlive_groups_and_looks():
    import gc
    import torch
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor, HipLinearGroup
    rng = np.random.default_rng(14)
    small, large = (HipContextTensor(codec.encode(weight_like(rng, rows, 1040))) for rows in (48, 700))
    pair = HipLinearGroup([small, HipContextTensor(codec.encode(weight_like(rng, 40, 1040)))])
    draw = lambda m: torch.from_numpy(bf16_words(rng.normal(0, 1, (m, 1040)))).view(torch.bfloat16).cuda()
    x1, x9 = draw(1), draw(9)
    step = lambda: [small.linear(x1), *pair.linear(x9), small.decode(check=False)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    group = HipLinearGroup([large, small])
    group.linear(x9)
    assert small.fused is not None and small.buffers["main_stream"].is_cuda
    gc.collect()
    torch.cuda.empty_cache()
    for _ in range(3):
        x1.copy_(draw(1)), x9.copy_(draw(9))
        eager = [v.clone() for v in step()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(captured, eager))
