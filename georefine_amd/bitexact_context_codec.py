"""BCTX frame container: exact BF16 word matrices <-> self-checking frames.

Mirrors the public surface of the reference module of the same name
(GCR/bitexact_context_codec.py: ``encode``:342, ``decode``:377, ``CodecError``:26,
``HEADER``:19, ``_labels``:183, ``_inflate_exact``:328 and the ``_encode_kind`` /
``_decode_kind`` / ``_pack6`` / ``_unpack6`` helpers the reference tests call).
The entropy coder itself is ``csrc/host_codec.cpp``.

Frame layout (little endian): 80-byte header ``BCTX``, version 1, mode
(0 raw 6-bit residual, 128 entropy-coded residual, 1 raw words), row/column
class counts, rows, cols, four section lengths, sha256 of the source words;
zlib(row labels ++ column labels); zlib(frequency tables); main rANS stream;
residual section; sha256 of everything before it.
"""
from __future__ import annotations

import ctypes
import hashlib
import os
import struct
import time
import zlib
from concurrent.futures import ThreadPoolExecutor

import numpy as np

from . import _native

MAGIC = b"BCTX"
VERSION = 1
HEADER = struct.Struct("<4sBBBBIIQQQQ32s")
MAX_WORDS = 0xFFFFFFFF
ROWS = {1, 4, 16, 64}
COLS = {1, 4, 16}
MAIN_VOCAB, RES_VOCAB, RES_CONTEXTS = 1024, 64, 1024


class CodecError(ValueError):
    """Invalid input or malformed frame."""


def _lib():
    return _native.codec()


def _input(words):
    """The matrix as contiguous little-endian uint16 words.  Accepted: two-dimensional arrays of
    16-bit integers (signed ones only where every value is a valid word's bit pattern read as
    unsigned, i.e. non-negative), non-empty, at most MAX_WORDS elements
    (GCR/bitexact_context_codec.py:172-180 accepts and rejects the same inputs)."""
    matrix = np.asarray(words)
    sixteen_bit_integers = matrix.dtype.kind in ("u", "i") and matrix.dtype.itemsize == 2
    if matrix.ndim != 2 or not sixteen_bit_integers:
        raise CodecError("expected a 2D uint16 word array")
    rows, cols = matrix.shape
    if rows == 0 or cols == 0 or rows * cols > MAX_WORDS:
        raise CodecError("invalid or oversized geometry")
    if matrix.dtype.kind == "i" and matrix.min() < 0:  # (an int16 cannot exceed 65535)
        raise CodecError("word outside uint16 range")
    return np.ascontiguousarray(matrix, dtype="<u2")


def _labels(a, nr, nc):
    """Quantile class of every row and column by summed magnitude bits.

    Sums are exact integers and ties keep index order, so labels do not depend
    on floating point (GCR/bitexact_context_codec.py:183-203)."""
    rows, cols = a.shape
    a = np.ascontiguousarray(a, dtype="<u2")
    row_sum, col_sum = np.empty(rows, dtype=np.uint64), np.empty(cols, dtype=np.uint64)
    if _lib().grf_bctx_sums(_native.ptr(a, ctypes.c_uint16), rows, cols, _native.ptr(row_sum, ctypes.c_uint64),
                            _native.ptr(col_sum, ctypes.c_uint64)):
        raise CodecError("class sums failed")

    def classes(total, k):
        rank = np.empty(len(total), dtype=np.uint64)
        rank[np.argsort(total, kind="stable")] = np.arange(len(total), dtype=np.uint64)
        return (rank * k // len(total)).astype(np.uint8)

    return classes(row_sum, nr), classes(col_sum, nc)


def _shape_of(kind, nr, nc):
    return (RES_VOCAB, RES_CONTEXTS) if kind else (MAIN_VOCAB, nr * nc)


def _u8(a):
    return np.ascontiguousarray(a, dtype=np.uint8)


def _encode_stream(lib, a, rc, cc, nr, nc, kind, freq):
    """The stream of one kind with the given frequency rows (bytes), as a view of the buffer it
    was written to."""
    rc, cc = _u8(rc), _u8(cc)
    rows = np.frombuffer(freq, dtype="<u4")
    buffer, begin = np.empty(2 * a.size + 8, dtype=np.uint8), ctypes.c_size_t()
    status = lib.grf_bctx_encode(_native.ptr(a, ctypes.c_uint16), a.shape[0], a.shape[1],
                                 _native.ptr(rc, ctypes.c_uint8), _native.ptr(cc, ctypes.c_uint8), nr, nc, kind,
                                 _native.ptr(rows, ctypes.c_uint32), _native.ptr(buffer, ctypes.c_uint8), buffer.size,
                                 ctypes.byref(begin))
    if status:
        raise CodecError(f"rANS encode failed ({status})")
    return memoryview(buffer)[begin.value:]


def _encode_kind(lib, a, rc, cc, nr, nc, kind):
    freq = _frequencies_kind(lib, a, rc, cc, nr, nc, kind)
    return freq, bytes(_encode_stream(lib, a, rc, cc, nr, nc, kind, freq))


def _frequencies_kind(lib, a, rc, cc, nr, nc, kind):
    vocab, nctx = _shape_of(kind, nr, nc)
    freq = np.zeros(nctx * vocab, dtype="<u4")
    rc, cc = _u8(rc), _u8(cc)
    status = lib.bcx_frequencies(_native.ptr(a, ctypes.c_uint16), a.size, a.shape[0], a.shape[1],
                                 _native.ptr(rc, ctypes.c_uint8), _native.ptr(cc, ctypes.c_uint8), nr, nc, kind,
                                 _native.ptr(freq, ctypes.c_uint32))
    if status:
        raise CodecError(f"frequency-only encode failed ({status})")
    return freq.tobytes()


def _decode_kind(lib, stream, freq, rc, cc, rows, cols, nr, nc, kind, main=None):
    choice = os.environ.get("GEOREFINE_CONTEXT_COMPACT_RANS")
    if choice not in (None, "0", "1"):
        raise CodecError("GEOREFINE_CONTEXT_COMPACT_RANS must be 0 or 1")
    fn = lib.bcx_decode_compact if choice == "1" else lib.bcx_decode
    vocab, nctx = _shape_of(kind, nr, nc)
    if len(freq) != nctx * vocab * 4:
        raise CodecError("frequency table length mismatch")
    table = np.frombuffer(freq, dtype="<u4").copy()
    n = rows * cols
    out = np.empty(n, dtype="<u2")
    rc, cc = _u8(rc), _u8(cc)
    data = np.frombuffer(bytes(stream), dtype=np.uint8) if len(stream) else np.zeros(1, np.uint8)
    ctx = None if main is None else np.ascontiguousarray(main, dtype="<u2").ravel()
    status = fn(_native.ptr(data, ctypes.c_uint8), len(stream), n, rows, cols, _native.ptr(rc, ctypes.c_uint8),
                _native.ptr(cc, ctypes.c_uint8), nr, nc, kind,
                _native.ptr(ctx, ctypes.c_uint16) if kind else _native.U16P(),
                _native.ptr(table, ctypes.c_uint32), _native.ptr(out, ctypes.c_uint16))
    if status:
        raise CodecError(f"rANS decode failed ({status})")
    return out if not kind else out.astype(np.uint8)


def _pack6(lib, a):
    out, size = _native.U8P(), ctypes.c_size_t()
    if lib.bcx_pack6(_native.ptr(a, ctypes.c_uint16), a.size, ctypes.byref(out), ctypes.byref(size)):
        raise CodecError("raw residual packing failed")
    try:
        return ctypes.string_at(out, size.value)
    finally:
        lib.bcx_free(out)


def _unpack6(lib, raw, n):
    out = np.empty(n, dtype="<u2")
    data = np.frombuffer(bytes(raw), dtype=np.uint8) if len(raw) else np.zeros(1, np.uint8)
    if lib.bcx_unpack6(_native.ptr(data, ctypes.c_uint8), len(raw), n, _native.ptr(out, ctypes.c_uint16)):
        raise CodecError("invalid raw residual stream")
    return out


def _inflate_exact(data, expected):
    """Inflate a section that must produce exactly ``expected`` bytes and nothing after."""
    inflater = zlib.decompressobj()
    try:
        raw = inflater.decompress(data, expected + 1)
        if len(raw) > expected or inflater.unconsumed_tail:
            raise CodecError("compressed section exceeds declared size")
        raw += inflater.flush()
    except zlib.error as exc:
        raise CodecError("invalid compressed section") from exc
    if len(raw) != expected or not inflater.eof or inflater.unused_data:
        raise CodecError("compressed section length/trailing data mismatch")
    return raw


def recombine(main, residual):
    """10-bit main symbol + 6-bit residual -> BF16 word (GCR/bitexact_context_codec.py:426)."""
    m = np.ascontiguousarray(main, dtype="<u2").ravel()
    r = np.ascontiguousarray(residual, dtype="<u2").ravel()
    out = np.empty(m.size, dtype="<u2")
    if m.size != r.size or _lib().grf_bctx_join(_native.ptr(m, ctypes.c_uint16), _native.ptr(r, ctypes.c_uint16),
                                                 m.size, _native.ptr(out, ctypes.c_uint16)):
        raise CodecError("symbol outside its alphabet")
    return out


def _sections(mode, nr, nc, r, c, meta, table, sy, rs, raw, dig):
    """A frame without its checksum, as the list of its parts."""
    return [HEADER.pack(MAGIC, VERSION, mode, nr, nc, r, c, len(meta), len(table), len(sy), len(rs), dig),
            meta, table, sy, rs, raw]


def _sealed(sections):
    sha = hashlib.sha256()
    for part in sections:
        sha.update(part)
    return b"".join((*sections, sha.digest()))


def encode(words, *, row_classes=16, col_classes=4, residual="auto"):
    """Encode a 2D BF16-bit-pattern array into a self-contained frame.

    Both residual forms are always produced and the shorter complete frame wins;
    a frame that is not shorter than the raw words falls back to mode 1.
    ``residual="raw6"`` (no counterpart in the reference's encoder, whose frames are the
    ``"auto"`` ones) writes the packed 6-bit residual section without trying the conditional
    stream: a mode-0 frame every decoder of the format takes, in about half the work.

    The two streams are serial chains that do not need each other: the conditional one is coded
    on a thread of its own, the words are hashed on another, and only the winner is assembled."""
    a = _input(words)
    if row_classes not in ROWS or col_classes not in COLS:
        raise CodecError("unsupported class count")
    if residual not in ("auto", "raw6"):
        raise CodecError("residual is \"auto\" or \"raw6\"")
    r, c = a.shape
    lib = _lib()
    raw = memoryview(a).cast("B")
    none = np.zeros(max(r, c), dtype=np.uint8)  # (the conditional stream's contexts are not the classes)

    classes = row_classes, col_classes

    with Beside(len(raw), workers=3) as beside:
        if residual == "auto":
            res_freq = beside.run(_frequencies_kind, lib, a, none[:r], none[:c], *classes, 1)
            res_stream = beside.run(lambda: _encode_stream(lib, a, none[:r], none[:c], *classes, 1, res_freq.result()))
        sha = beside.run(lambda: hashlib.sha256(raw).digest())
        rc, cc = _labels(a, *classes)
        main_freq = _frequencies_kind(lib, a, rc, cc, *classes, 0)
        table = beside.run(zlib.compress, main_freq, 6)
        if residual == "auto":
            both = beside.run(lambda: zlib.compress(main_freq + res_freq.result(), 6))
        packed = beside.run(_pack6, lib, a)
        meta = zlib.compress(rc.tobytes() + cc.tobytes(), 6)
        main_stream = _encode_stream(lib, a, rc, cc, *classes, 0, main_freq)
        dig, table, packed = sha.result(), table.result(), packed.result()
        fixed = HEADER.size + len(meta) + len(main_stream) + 32
        size = fixed + len(table) + len(packed)
        if residual == "auto":
            both, res_stream = both.result(), res_stream.result()
            conditional_size = fixed + len(both) + len(res_stream)
    if min(size, conditional_size if residual == "auto" else size) >= HEADER.size + len(raw) + 32:
        return _sealed(_sections(1, row_classes, col_classes, r, c, b"", b"", b"", b"", raw, dig))
    if residual == "auto" and conditional_size < size:
        return _sealed(_sections(128, row_classes, col_classes, r, c, meta, both, main_stream, res_stream, b"", dig))
    return _sealed(_sections(0, row_classes, col_classes, r, c, meta, table, main_stream, packed, b"", dig))


def parse(frame):
    """Validate everything that does not need entropy decoding and split the frame.

    Returns a dict: ``mode nr nc shape digest`` and, for coded modes, ``rows columns
    main_freq [residual_freq] main_stream residual_stream``; for mode 1 ``raw``."""
    frame = _frame_bytes(frame)
    if not _frame_digests(frame)[0]:
        raise CodecError("frame checksum mismatch")
    info = _split(frame)
    for name in ("main_stream", "residual_stream"):
        if name in info:
            info[name] = bytes(info[name])
    return info


def _frame_bytes(frame):
    if not isinstance(frame, (bytes, bytearray, memoryview)) or len(frame) < HEADER.size:
        raise CodecError("short frame")
    return bytes(frame)


def _frame_digests(frame):
    """(whether the frame's own checksum holds, SHA-256 of the whole frame in hex): one pass."""
    if len(frame) < HEADER.size + 32:
        return False, None
    sha = hashlib.sha256(memoryview(frame)[:-32])
    own = sha.digest() == frame[-32:]
    sha.update(frame[-32:])
    return own, sha.hexdigest()


def _split(frame):
    """``parse`` without the checksum; the streams are views of the frame."""
    magic, ver, mode, nr, nc, r, c, ml, tl, sl, dl, dig = HEADER.unpack_from(frame)
    if magic != MAGIC or ver != VERSION or nr not in ROWS or nc not in COLS:
        raise CodecError("unsupported frame header")
    n = r * c
    if not r or not c or n > MAX_WORDS:
        raise CodecError("invalid geometry")
    info = dict(mode=mode, nr=nr, nc=nc, shape=(r, c), digest=dig)
    end = HEADER.size + ml + tl + sl + dl
    if mode == 1:
        if ml or tl or sl or dl or len(frame) != end + 2 * n + 32:
            raise CodecError("invalid raw frame length")
        raw = memoryview(frame)[end:-32]
        if hashlib.sha256(raw).digest() != dig:
            raise CodecError("raw checksum mismatch")
        info["raw"] = np.frombuffer(raw, dtype="<u2").copy().reshape(r, c)
        return info
    if mode not in (0, 128) or len(frame) != end + 32:
        raise CodecError("invalid frame mode/length")
    at = HEADER.size
    labels = _inflate_exact(frame[at:at + ml], r + c)
    at += ml
    main_bytes = nr * nc * MAIN_VOCAB * 4
    tables = _inflate_exact(frame[at:at + tl], main_bytes + (RES_CONTEXTS * RES_VOCAB * 4 if mode == 128 else 0))
    at += tl
    info["rows"] = np.frombuffer(labels[:r], dtype=np.uint8).copy()
    info["columns"] = np.frombuffer(labels[r:], dtype=np.uint8).copy()
    if info["rows"].max(initial=0) >= nr or info["columns"].max(initial=0) >= nc:
        raise CodecError("class outside declared range")
    info["main_freq"] = np.frombuffer(tables[:main_bytes], dtype="<u4").copy().reshape(nr * nc, MAIN_VOCAB)
    if mode == 128:
        info["residual_freq"] = np.frombuffer(tables[main_bytes:], dtype="<u4").copy().reshape(RES_CONTEXTS, RES_VOCAB)
    info["main_stream"] = memoryview(frame)[at:at + sl]
    info["residual_stream"] = memoryview(frame)[at + sl:at + sl + dl]
    return info


class _Now:
    """A result that was computed at once (what a pool's future is for small inputs)."""

    def __init__(self, value):
        self.value = value

    def result(self):
        return self.value


class Beside:
    """One thread for work beside the caller's (hashing, a second stream), for as long as the
    ``with`` block; inputs under ``BESIDE_FROM`` bytes are not worth one and run at once."""

    BESIDE_FROM = 1 << 18

    def __init__(self, nbytes, workers=1):
        self.pool = ThreadPoolExecutor(max_workers=workers) if nbytes >= self.BESIDE_FROM else None

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        if self.pool is not None:
            self.pool.shutdown()

    def run(self, fn, *args):
        return self.pool.submit(fn, *args) if self.pool is not None else _Now(fn(*args))


def _sha_following(words, progress):
    """SHA-256 of ``words`` while they are written: ``progress[0]`` of them are final.  None if
    the walk gave up (a count beyond the end)."""
    sha, view, done, step = hashlib.sha256(), memoryview(words).cast("B"), 0, 1 << 17
    while done < words.size:
        ready = int(progress[0])
        if ready > words.size:
            return None
        if ready - done < min(step, words.size - done):
            time.sleep(1e-4)
            continue
        sha.update(view[2 * done:2 * ready])
        done = ready
    return sha.digest()


def _decode_failed(status):
    """The message of a failed walk as ``bcx_decode`` reports it: 3 internal, 2 anything else."""
    return f"rANS decode failed ({3 if status in (5, 6) else 2})"


def read_words(frame, stride=0, failed=_decode_failed):
    """A whole frame decoded and checked against its own checksum: the dict of ``parse`` with
    ``words`` (one-dimensional), ``words_digest`` and ``frame_sha256``; with ``stride`` also
    the main stream's index, ``main_states`` and ``main_offsets``.  The walk runs on the caller's
    thread (and one in the library); the frame and the finished words are hashed beside it.
    ``failed``: the message of a walk's status (``grf_bctx_words``, whichever stream's)."""
    frame = _frame_bytes(frame)
    with Beside(len(frame)) as beside:
        digests = beside.run(_frame_digests, frame)
        try:
            info = _split(frame)
            if info["mode"] == 1:
                info["words"], info["words_digest"] = info["raw"].reshape(-1), info["digest"]
            else:
                _walk(info, stride, failed, beside)
        except CodecError:
            if not digests.result()[0]:
                raise CodecError("frame checksum mismatch") from None
            raise
        own, info["frame_sha256"] = digests.result()
        if not own:
            raise CodecError("frame checksum mismatch")
        if not isinstance(info["words_digest"], bytes):
            info["words_digest"] = info["words_digest"].result()
    return info


def _walk(info, stride, failed, beside):
    r, c = info["shape"]
    words = info["words"] = np.empty(r * c, dtype="<u2")
    progress = np.zeros(1, dtype=np.uint64)
    states = offsets = None
    if stride:
        states, offsets = (np.empty(-(-words.size // stride), dtype=np.uint32) for _ in range(2))
        info["main_states"], info["main_offsets"] = states, offsets
    p = lambda a, t: _native.ptr(a, t) if a is not None else ctypes.POINTER(t)()
    digest, status = None, -1
    try:
        if beside.pool is not None:  # a thread hashes behind the walk; without one the hash follows it
            digest = beside.run(_sha_following, words, progress)
        streams = [np.frombuffer(s, dtype=np.uint8) if len(s) else np.zeros(1, np.uint8)
                   for s in (info["main_stream"], info["residual_stream"])]
        status = _lib().grf_bctx_words(
            p(streams[0], ctypes.c_uint8), len(info["main_stream"]), r, c, p(info["rows"], ctypes.c_uint8),
            p(info["columns"], ctypes.c_uint8), info["nr"], info["nc"], p(info["main_freq"], ctypes.c_uint32), stride,
            p(states, ctypes.c_uint32), p(offsets, ctypes.c_uint32), p(streams[1], ctypes.c_uint8),
            len(info["residual_stream"]), p(info.get("residual_freq"), ctypes.c_uint32), p(words, ctypes.c_uint16),
            p(progress, ctypes.c_uint64))
    finally:
        if status:  # whatever went wrong, from the thread's start on: nothing follows the walk any more
            progress[0] = np.uint64(0xFFFFFFFFFFFFFFFF)
    if status:
        raise CodecError("invalid raw residual stream" if status == 33 else failed(status % 16))
    info["words_digest"] = digest if digest is not None else hashlib.sha256(words).digest()


def decode(frame):
    """Decode a complete frame on the host and verify the source checksum."""
    if os.environ.get("GEOREFINE_CONTEXT_COMPACT_RANS") not in (None, "0", "1"):
        raise CodecError("GEOREFINE_CONTEXT_COMPACT_RANS must be 0 or 1")
    info = read_words(frame)
    if info["words_digest"] != info["digest"]:
        raise CodecError("decoded checksum mismatch")
    return info["words"].reshape(info["shape"])
