"""A tensor that is held as planes stays so whatever is looked at, and a group leaves its members as they are
(no GPU: device calls are stand-ins, and the arrays are the host's)."""
import contextlib
import gc
import threading
import types
import weakref

import numpy as np
import pytest
import torch

from conftest import bf16_words, weight_like
from georefine_amd import _planes
from georefine_amd import bitexact_context_codec as codec
from georefine_amd import bitexact_context_gpu as gpu
from georefine_amd import bitexact_predictive_codec as predictive
from georefine_amd import bitexact_predictive_gpu as pgpu


class _HostPlanes(_planes.Planes):
    """Planes that keep the words they were laid out from."""

    def __init__(self, words):
        self.rows, self.cols = words.shape
        exponents = (words.int() >> 7 & 255).long()
        held = torch.zeros(self.rows, 256, dtype=torch.int64).scatter_add_(1, exponents, torch.ones_like(exponents))
        listed = words.numel() - int(held.unfold(1, _planes.EXPONENTS, 1).sum(2).amax(1).sum())
        self.words, self.nbytes, self.address = words, _planes.plane_bytes(*words.shape) + 4 * listed, 0

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
    for cls in (gpu.HipContextTensor, pgpu.HipPredictiveTensor):
        on_device = cls.decode

        def decode(self, *args, general=False, on_device=on_device, **kw):
            return on_device(self, *args, general=general, **kw) if general or self._planes is None else self._planes.words.view(torch.bfloat16)

        monkeypatch.setattr(cls, "decode", decode)


def _context(rows, cols=1024, seed=1, **kw):
    return gpu.HipContextTensor(codec.encode(weight_like(np.random.default_rng(seed), rows, cols)), device="cpu", **kw)


def _predictive(rows=512, cols=1024):
    rng = np.random.default_rng(2)
    target = weight_like(rng, rows, cols)
    near = bf16_words((target.astype(np.uint32) << 16).view(np.float32) + rng.normal(0, 0.002, (rows, cols)).astype(np.float32))
    return pgpu.HipPredictiveTensor(predictive.encode(target, near), near, device="cpu")


@pytest.mark.parametrize("make", [lambda: _context(512), _predictive], ids=["context", "predictive"])
def test_looking_at_the_walks_arrays_leaves_what_products_run_on(make):
    t = make()
    planes, held = t._planes, t.resident_bytes
    assert planes is not None and "buffers" not in vars(t)
    buffers, fused = t.buffers, t.fused
    assert t._planes is planes and fused is not None and t.fusable
    assert t.buffers is buffers and t.fused is fused  # the same arrays from then on: their addresses stay good
    arrays = sum(a.numel() * a.element_size() for a in buffers.values())
    assert t.resident_bytes >= held + arrays  # what both take
    other = t.clone()
    assert "buffers" not in vars(other) and other.resident_bytes == held and other._planes is not planes
    assert other.buffers["main_stream"] is not buffers["main_stream"]
    assert all(torch.equal(other.buffers[name], array) for name, array in buffers.items() if array.dtype is torch.uint8)


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


def test_another_thread_never_sees_half_of_the_walks_attributes(monkeypatch):
    t, within, go, seen = _context(512), threading.Event(), threading.Event(), []
    bind = gpu.HipContextTensor._bind

    def slow(self):
        within.set()
        assert go.wait(60)
        bind(self)

    monkeypatch.setattr(gpu.HipContextTensor, "_bind", slow)
    first = threading.Thread(target=lambda: t.buffers)
    first.start()
    assert within.wait(60)
    second = threading.Thread(target=lambda: seen.append(t.fused))
    second.start()
    second.join(0.2)
    go.set()
    first.join(), second.join()
    assert seen[0] is not None and seen[0] is t.fused


def test_a_predictive_frame_is_decoded_once_whatever_it_is_held_as(monkeypatch):
    """One whose words the planes would mostly list stays a frame, and is not read a second time for it."""
    rng, walks = np.random.default_rng(5), []
    spread = (rng.integers(0, 2, (512, 1024)) << 15 | rng.integers(60, 180, (512, 1024)) << 7 | rng.integers(0, 128, (512, 1024))).astype(np.uint16)
    near = spread ^ rng.integers(0, 4, spread.shape).astype(np.uint16)
    counted = pgpu._checkpoints
    monkeypatch.setattr(pgpu, "_checkpoints", lambda *a: walks.append(len(a[0])) or counted(*a))
    monkeypatch.setattr(pgpu.HipPredictiveTensor, "_bins", lambda self, ref: (torch.zeros(1, dtype=torch.int32), 0))
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device: None)
    for target, as_planes in ((spread, False), (weight_like(rng, 512, 1024), True)):
        frame = predictive.encode(target, near)
        streams = 1 if frame[5] == 0 else 2
        walks.clear()
        t = pgpu.HipPredictiveTensor(frame, near, device="cpu")
        assert (t._planes is not None) == as_planes and len(walks) <= streams, (as_planes, walks)
        # bytes of the host's that a tensor keeps, for as long as it lives
        assert t.host_bytes == (near.size // 2 + len(t._kept["meta"]) + len(t._kept["table"]) if as_planes else 0)
