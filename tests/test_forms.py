"""A group leaves its members in the form that they are held in (no GPU: device calls are stand-ins, and the
arrays are the host's)."""
import gc
import types
import weakref

import numpy as np
import pytest
import torch

from conftest import weight_like
from georefine_amd import _planes
from georefine_amd import bitexact_context_codec as codec
from georefine_amd import bitexact_context_gpu as gpu


class _HostPlanes(_planes.Planes):
    """Planes that keep the words they were laid out from."""

    def __init__(self, words):
        self.rows, self.cols = words.shape
        self.words, self.nbytes, self.address = words, words.numel() * 3 // 2, 0

    @classmethod
    def of_words(cls, words, launch):
        return cls(words)

    def clone(self):
        return _HostPlanes(self.words.clone())


@pytest.fixture(autouse=True)
def host(monkeypatch):
    stream = types.SimpleNamespace(synchronize=lambda: None, cuda_stream=None)
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: stream)
    monkeypatch.setattr(_planes, "Planes", _HostPlanes)
    monkeypatch.setattr(gpu, "device_index", lambda device: 0)
    monkeypatch.setattr(gpu, "_residual_form", lambda groups, to_pairs: groups)


def _context(rows, cols=1024, seed=1, **kw):
    return gpu.HipContextTensor(codec.encode(weight_like(np.random.default_rng(seed), rows, cols)), device="cpu", **kw)


def test_a_group_with_a_large_member_keeps_the_small_ones_arrays():
    large, small = _context(512), _context(48)
    assert small._planes is None
    before, main, held = small.buffers, weakref.ref(small.buffers["main_stream"]), small.resident_bytes
    alone = gpu.HipLinearGroup([small, _context(40, seed=3)])
    frames = alone._arrays("gemm", [torch.empty(1)] * 2, None)[0]
    gpu.HipLinearGroup([large, small])
    assert small._planes is None and small.buffers is before and small.resident_bytes == held
    del before
    gc.collect()
    assert main() is not None and main() is small.buffers["main_stream"]
    assert frames[0].contents.main_bytes == main().data_ptr()  # what the first group launches with
