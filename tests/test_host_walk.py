"""The host coder's walks against the oracle where their cuts fall: runs at row ends and marks, the
last symbols of a stream, contexts that are one symbol, symbols behind a bucket's boundary."""
import ctypes
import hashlib
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from georefine_amd import _native
from georefine_amd import bitexact_context_codec as codec
from georefine_amd.bitexact_context_gpu import checkpoints, index_frame


def _words(kind, rows, cols):
    rng = np.random.default_rng(rows * 1009 + cols)
    if kind == "weights":  # a few dozen symbols per context, as coded weights have
        w = (rng.standard_normal((rows, cols)) * 0.02 * rng.lognormal(0, 0.5, (rows, 1))).astype(np.float32)
        return (w.view(np.uint32) >> 16).astype(np.uint16)
    if kind == "flat":  # every symbol in every context: several a bucket
        return rng.integers(0, 65536, (rows, cols), dtype=np.uint16)
    return np.where(rng.random((rows, cols)) < 0.01, 0x4000, 0x3F80).astype(np.uint16)


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 63), (64, 65), (5, 4099), (300, 300)])
@pytest.mark.parametrize("kind", ["weights", "flat", "two"])
def test_walks_match_the_oracle(oracle, kind, rows, cols):
    words = _words(kind, rows, cols)
    rc, cc = codec._labels(words, 4, 4)
    for stream_kind in (0, 1):
        main = ((words >> 5) & 0x3FF).ravel() if stream_kind else None
        freq, stream = codec._encode_kind(codec._lib(), words, rc, cc, 4, 4, stream_kind)
        table = np.frombuffer(freq, dtype="<u4").reshape((1024, 64) if stream_kind else (16, 1024))
        want_freq, want_stream = oracle.bcx_encode_kind(words, rc, cc, 4, 4, stream_kind)
        assert np.array_equal(table.ravel(), np.asarray(want_freq).ravel()) and stream == bytes(want_stream)
        for stride in (1, 64, rows * cols):
            got = checkpoints(stream, table, rc, cc, (rows, cols), 4, 4, stride, main)
            want = oracle.bcx_checkpoint(stream, table, rc, cc, rows, cols, 4, 4, stride, main)
            assert all(np.array_equal(a, b) for a, b in zip(got, want))


_NO_MEMORY_IN_THE_WALK = """
import sys
import numpy as np
from georefine_amd import bitexact_context_codec as codec
rng = np.random.default_rng(0)
frame = codec.encode((rng.integers(0, 4, (600, 640)) << 7 | rng.integers(0, 64, (600, 640))).astype(np.uint16))
assert frame[5] != 1 and len(frame) >= codec.Beside.BESIDE_FROM  # hashed beside the walk

class Numpy:  # numpy, but stream views made inside the walk find no memory
    def __getattr__(self, name):
        return getattr(np, name)
    def frombuffer(self, *args, **kw):
        if "_walk" in (sys._getframe(1).f_code.co_name, sys._getframe(2).f_code.co_name):
            raise MemoryError
        return np.frombuffer(*args, **kw)

codec.np = Numpy()
try:
    codec.decode(frame)
except MemoryError:
    print("raised")
"""


def test_an_exception_beside_the_hashing_thread_reaches_the_caller():
    """Whatever is raised once the thread that follows the walk may run ends that thread too (in a
    process of its own: a thread left behind would keep this one from ending)."""
    done = subprocess.run([sys.executable, "-c", _NO_MEMORY_IN_THE_WALK], cwd=Path(__file__).resolve().parent.parent,
                          capture_output=True, text=True, timeout=60)
    assert done.stdout == "raised\n", done.stderr[-2000:]


def _one_stream_after_the_other(frame, index):
    """What a frame's walk reports, stream by stream through the entry points the reference binds."""
    info = codec.parse(frame)
    (r, c), nr, nc = info["shape"], info["nr"], info["nc"]
    tables = info["main_freq"], info.get("residual_freq")
    classes = info["rows"], info["columns"]
    try:
        main = (checkpoints(info["main_stream"], tables[0], *classes, (r, c), nr, nc, 1024)[2] if index else
                codec._decode_kind(codec._lib(), info["main_stream"], tables[0].tobytes(), *classes, r, c, nr, nc, 0))
        if tables[1] is None:
            residual = codec._unpack6(codec._lib(), info["residual_stream"], r * c)
        elif index:
            residual = checkpoints(info["residual_stream"], tables[1], *classes, (r, c), nr, nc, 1024, main)[2]
        else:
            residual = codec._decode_kind(codec._lib(), info["residual_stream"], tables[1].tobytes(), *classes, r, c, nr,
                                          nc, 1, main)
    except codec.CodecError as exc:
        return str(exc)
    words = codec.recombine(main, residual)
    if hashlib.sha256(words.tobytes()).digest() != info["digest"]:
        return "indexed source checksum mismatch" if index else "decoded checksum mismatch"
    return words.reshape(r, c)


def _with_streams(frame, main=None, residual=None):
    """The frame with another stream or two, sealed with a checksum that holds."""
    header = list(codec.HEADER.unpack_from(frame))
    at = codec.HEADER.size + header[7] + header[8]
    streams = [frame[at:at + header[9]], frame[at + header[9]:at + header[9] + header[10]]]
    for i, change in enumerate((main, residual)):
        if change is not None:
            streams[i] = change(streams[i])
            header[9 + i] = len(streams[i])
    return codec._sealed([codec.HEADER.pack(*header), frame[codec.HEADER.size:at], *streams])


def _flipped(at):
    return lambda s: s[:at] + bytes([s[at] ^ 0x55]) + s[at + 1:]


_DAMAGE = {
    "whole": None, "head": _flipped(3), "early": _flipped(9), "middle": lambda s: _flipped(len(s) // 2)(s),
    "last": lambda s: _flipped(len(s) - 1)(s), "cut": lambda s: s[:-3], "half": lambda s: s[:len(s) // 2],
    "longer": lambda s: s + b"\0\0", "no head": lambda s: s[:3], "empty": lambda s: b"",
}


@pytest.mark.parametrize("rows,cols", [(37, 210), (700, 511)])  # the second: two threads in the library, one beside it
@pytest.mark.parametrize("mode", [0, 128])
def test_damaged_streams_are_reported_as_by_one_walk_after_the_other(rows, cols, mode):
    rng = np.random.default_rng(rows + mode)
    fields = rng.integers(0, 64 if mode == 0 else 3, (rows, cols))
    main = rng.geometric(0.1, (rows, cols)) % 60
    words = (main << 5 | (fields & 31) | (fields & 32) << 10).astype(np.uint16)
    frame = codec.encode(words, residual="raw6" if mode == 0 else "auto")
    assert frame[5] == mode and (words.size >= 1 << 18) == (rows > 100)
    for stream in ("main", "residual"):
        for name, damage in _DAMAGE.items():
            broken = _with_streams(frame, **{stream: damage})
            for index in (False, True):
                want = _one_stream_after_the_other(broken, index)
                try:
                    got = codec.decode(broken) if not index else index_frame(broken, 1024)
                except codec.CodecError as exc:
                    assert str(exc) == want, (stream, name, index)
                else:
                    assert isinstance(want, np.ndarray), (stream, name, index)
                    assert index or np.array_equal(got, want)


def test_a_stream_of_any_length_is_decoded_and_one_past_32_bits_is_not_indexed():
    """The index holds byte offsets of 32 bits; words alone need none.  (The length is claimed, not
    allocated: the walk ends with its last symbol, finds the stream's end elsewhere and says so.)"""
    n = 64
    buffer = np.full(4 * n + 64, 0x80, dtype=np.uint8)
    classes, freq = np.zeros(n, dtype=np.uint8), np.zeros(1024, dtype=np.uint32)
    freq[:2] = 32768
    packed, words = np.zeros(n * 6 // 8, dtype=np.uint8), np.zeros(n, dtype=np.uint16)
    states, offsets = np.zeros(n, dtype=np.uint32), np.zeros(n, dtype=np.uint32)
    p = lambda a, t: _native.ptr(a, t)
    for stride, status in ((0, 3), (1, 1)):
        assert codec._lib().grf_bctx_words(
            p(buffer, ctypes.c_uint8), (1 << 32) + 5, 1, n, p(classes, ctypes.c_uint8), p(classes, ctypes.c_uint8), 1, 1,
            p(freq, ctypes.c_uint32), stride, p(states, ctypes.c_uint32), p(offsets, ctypes.c_uint32),
            p(packed, ctypes.c_uint8), packed.size, ctypes.POINTER(ctypes.c_uint32)(), p(words, ctypes.c_uint16),
            ctypes.POINTER(ctypes.c_uint64)()) == status
