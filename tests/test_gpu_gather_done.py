"""A gather tells the host that it is over: every count of rows around the counters', ids that are refused and rows that do
not decode, calls that share words and counters over threads and streams, and a wait that gives up."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tensor(rows=300, cols=64 * 30, seed=3, **options):
    from georefine_amd import bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    rng = np.random.default_rng(seed)
    words = (rng.choice([0x3C00, 0x3C20, 0x3D00], (rows, cols)) | rng.integers(0, 32, (rows, cols))).astype(np.uint16)
    return HipContextTensor(codec.encode(words), **options), words


@pytest.mark.parametrize("count", [1, 2, 31, 32, 33, 63, 65, 777, 1025])
def test_counters_return_to_zero(count):
    import torch
    from georefine_amd import _hip_abi
    t, words = _tensor()
    t.gather_rows(torch.tensor([0]))
    ids = torch.from_numpy(np.random.default_rng(count).integers(0, 300, count))
    ids[count // 2] = 299
    counters = torch.zeros(_hip_abi.GATHER_COUNTER_BYTES // 4, dtype=torch.int32, device="cuda")
    word = torch.zeros(1, dtype=torch.int32, pin_memory=True)
    out = torch.empty((count, t.shape[1]), device="cuda", dtype=torch.int16)
    for bad in (None, 300, None):
        on_device = ids.clone()
        if bad is not None:
            on_device[-1] = bad
        on_device = on_device.cuda()
        word[0] = 0
        t._launch(t._lib.grf_bctx_gather_rows_done, ctypes.byref(t.fused), *t._gather, t.buffers["rows"].data_ptr(), on_device.data_ptr(),
                  count, out.data_ptr(), word.data_ptr(), word.data_ptr(), counters.data_ptr(), word.data_ptr())
        torch.cuda.synchronize()
        assert word.item() == _hip_abi.GATHER_DONE | (_hip_abi.ERR_INDEX if bad else 0) and not counters.any()
    assert np.array_equal(out.cpu().numpy().view(np.uint16), words[ids.numpy()])


@pytest.mark.parametrize("segment", [16, 32, 64])
@pytest.mark.parametrize("count", [1, 777, 3999, 4000])
def test_lookups_that_are_polled_for_and_that_are_not(segment, count, form):
    import torch
    t, words = _tensor(fused_segment=segment)
    assert (t._planes is not None) == (form == "planes") and t.fused.seg_len == segment
    ids = torch.from_numpy(np.random.default_rng(count).integers(0, 300, count))
    want, on_device = words[ids.numpy()], ids.cuda()
    for options in ({}, {"check": False}, {"check": False, "validate": False}):
        got = t.gather_rows(on_device, **options)
        assert np.array_equal(got.view(torch.int16).cpu().numpy().view(np.uint16), want), options
    for bad in (300, -1):
        on_device[count // 2] = bad
        for options in ({}, {"check": False}):
            with pytest.raises(IndexError):
                t.gather_rows(on_device, **options)
        clamped = t.gather_rows(on_device, check=False, validate=False)[count // 2]
        assert np.array_equal(clamped.view(torch.int16).cpu().numpy().view(np.uint16), words[299 if bad > 0 else 0])


@pytest.mark.parametrize("count", [1, 40])
def test_a_refused_row_keeps_its_output(count):
    import torch
    from georefine_amd import _hip_abi
    t, words = _tensor()
    t.gather_rows(torch.tensor([0]))
    ids = torch.arange(count)
    ids[count // 2] = 300
    on_device, word = ids.cuda(), torch.zeros(1, dtype=torch.int32, pin_memory=True)
    counters = torch.zeros(_hip_abi.GATHER_COUNTER_BYTES // 4, dtype=torch.int32, device="cuda")
    for told in (False, True):
        out = torch.full((count, t.shape[1]), 7, device="cuda", dtype=torch.int16)
        about = (ctypes.byref(t.fused), *t._gather, t.buffers["rows"].data_ptr(), on_device.data_ptr(), count, out.data_ptr(), word.data_ptr(),
                 word.data_ptr())
        word[0] = 0
        t._launch(*(t._lib.grf_bctx_gather_rows_done, *about, counters.data_ptr(), word.data_ptr()) if told else
                  (t._lib.grf_bctx_gather_rows, *about))
        torch.cuda.synchronize()
        assert word.item() == _hip_abi.ERR_INDEX | (_hip_abi.GATHER_DONE if told else 0)
        got = out.cpu().numpy().view(np.uint16)
        assert (got[count // 2] == 7).all()
        assert all(np.array_equal(got[k], words[k]) for k in range(count) if k != count // 2)


@pytest.mark.parametrize("spin", [0, 100])
def test_threads_on_streams_of_their_own(spin, form, monkeypatch):
    import torch
    from georefine_amd import bitexact_context_gpu as gpu
    monkeypatch.setattr(gpu, "GATHER_SPIN_US", spin)  # 0: every call waits for its stream
    t, words = _tensor()
    t.gather_rows(torch.tensor([0]))
    wrong = []

    def serve(seed):
        rng = np.random.default_rng(seed)
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                ids = torch.from_numpy(rng.integers(0, 300, int(rng.integers(1, 200)))).cuda()
                if not np.array_equal(t.gather_rows(ids).view(torch.int16).cpu().numpy().view(np.uint16), words[ids.cpu().numpy()]):
                    wrong.append(seed)

    threads = [threading.Thread(target=serve, args=(i,)) for i in range(4)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert not wrong


def test_refused_on_the_host():
    from georefine_amd import _native
    lib = _native.hip()
    assert lib.grf_bctx_gather_rows_done(None, 4, 16, None, None, 0, None, None, None, None, None, None) != 0
    word = ctypes.c_int32(0)
    assert lib.grf_wait_word(ctypes.addressof(word), 1, 10) == 0
    word.value = 3
    assert lib.grf_wait_word(ctypes.addressof(word), 1, 0) == 1 and lib.grf_wait_word(None, 1, 0) == 0
    assert lib.grf_take_word(ctypes.addressof(word), 4, 10) == 0 and word.value == 3
    assert lib.grf_take_word(ctypes.addressof(word), 1, 0) == 3 and word.value == 0 and lib.grf_take_word(None, 1, 0) == 0
