"""Indexed device decoding of PPCX frames on MI355X.

``_read_frame`` and ``HipPredictiveTensor`` keep the contract of the reference's
``_read_frame`` / ``CudaPredictiveTensor`` (GCR/bitexact_predictive_gpu.py:87-136 and
:138-174): ``factory(frame, reference_uint16_numpy, stride=..., device=...)``, then
``shape``, ``frame_sha256``, ``source_sha256``, ``resident_bytes`` and
``decode(reference_bf16_device, check=)``.  The reference words are an input of every
decode: the kernel derives each symbol's context from the reference word at the same
position (sign alignment per row, ordinal key, threshold bin).  A tensor that keeps its contexts
needs no reference in a call; its words are then held as planes (``_planes``: 96 rows of 4096 x 4096
23.5 us where the walk takes 40.8, in 24 MB where that takes 34), small ones as the frame's arrays.
"""
from __future__ import annotations

import ctypes
import hashlib
import math
import os

import numpy as np

from . import _fused, _hip_abi, _native, _planes, _tables
from . import bitexact_predictive_codec as codec


def _ptr(a, t):
    return a.ctypes.data_as(ctypes.POINTER(t))


def _checkpoints(stream, ctx, freq, vocab, stride):
    """(states, offsets, symbols) of one stream via ``ppcx_checkpoint``."""
    ctx = np.ascontiguousarray(ctx, dtype="<u2")
    freq = np.ascontiguousarray(freq, dtype="<u4")
    n = len(ctx)
    states = np.empty((n + stride - 1) // stride, dtype="<u4")
    offsets = np.empty_like(states)
    symbols = np.empty(n, dtype="<u2")
    data = np.frombuffer(stream, dtype=np.uint8)
    backend = os.environ.get("BITEXACT_PREDICTIVE_FAST_INDEX", "0")
    if backend not in ("0", "1"):
        raise codec.CodecError("BITEXACT_PREDICTIVE_FAST_INDEX must be 0 or 1")
    lib = _native.codec()
    fn = lib.ppcx_checkpoint_binary if backend == "1" else lib.ppcx_checkpoint
    status = fn(_ptr(data, ctypes.c_uint8), len(data), n, _ptr(ctx, ctypes.c_uint16), freq.size // vocab, vocab,
                _ptr(freq, ctypes.c_uint32), stride, _ptr(states, ctypes.c_uint32), _ptr(offsets, ctypes.c_uint32),
                _ptr(symbols, ctypes.c_uint16))
    if status:
        raise codec.CodecError(f"PPCX checkpoint validation failed ({status})")
    return states, offsets, symbols


# Sixteen bin contexts share the lookup bytes.  A wave scans on whenever one of its 64 lanes meets
# a bucket's minority symbol: 35 % of the steps with 1 KiB per context, 21 % with 2 KiB, 12 % with
# 4 KiB.  At 64 KiB one workgroup of sixteen waves has a compute unit to itself instead of two of
# twelve, and still wins for products on the matrix cores (16 / 32 / 64 KiB in all, us: 3000 x 4096
# at 96 rows 36.4 / 32.6 / 31.9, 5120 x 17408 156 / 142 / 135, 512 x 1024 at 64 rows 15.8 / 15.2 / 15.1), except
# where three of eight waves at 16 KiB do (_fused.fewer_lookups_pay).
# One row and decode() take 32 KiB where those are faster (FramePlan.for_vector_alus).  The tensor keeps
# every lookup it uses, half and a quarter MiB more.
_LUT_BUDGET, _WALK_LUT_BUDGET = ((int(os.environ["GEOREFINE_FUSED_LUT_BYTES"]),) * 2
                                 if "GEOREFINE_FUSED_LUT_BYTES" in os.environ else (64 * 1024, 32 * 1024))
_MATRIX_LUT_BUDGET = 16 * 1024


def _word_image(main):
    """Bits of a main symbol in the BF16 word: sign, exponent, mantissa bits 6..5
    (GCR/bitexact_predictive_codec.py:248)."""
    return ((main & 1024) << 5) | (((main >> 2) & 255) << 7) | ((main & 3) << 5)


def _fused_segment(shape, segment=None):
    """Segment length for the tile walker (a multiple of 32 that divides the row length)."""
    r, c = shape
    if c % 32:
        raise _fused.FusedUnsupported("row length is not a multiple of 32")
    order = [32, 64, 128, 256] if r * c < _fused.SMALL_MATRIX else [64, 128, 32, 256]
    seg_len = next((s for s in ([segment] if segment else []) + order if s and s % 32 == 0 and c % s == 0), None)
    if seg_len is None:
        raise _fused.FusedUnsupported("no segment length divides the row length")
    return seg_len


def _read_frame(frame, reference, stride, *, fused=False, fused_segment=None, planes=False):
    """Parse, validate and index a frame against its reference words.  With ``fused`` the
    result also carries ``fused_plan`` (or ``fused_reason``) with ``walk_plan``, the same with the lookups
    of the vector-ALU launches, and keeps the residuals in the packed 5-bit form whatever the
    frame's mode (``resident_mode`` 0).  With ``planes`` as well, a frame that is better held so gives its words and no index
    (``_words_of``)."""
    if not isinstance(frame, (bytes, bytearray, memoryview)):
        raise codec.CodecError("frame must be bytes")
    info = codec.parse(frame, reference)
    r, c = info["shape"]
    n = r * c
    target_hash = info["target_sha256"]
    result = dict(shape=(r, c), mode=info["mode"], frame_bytes=len(frame),
                  frame_sha256=hashlib.sha256(bytes(frame)).hexdigest(), source_sha256=target_hash.hex(),
                  target_sha256=target_hash.hex(), reference_sha256=info["reference_sha256"].hex())
    if info["mode"] == 2:
        target = np.frombuffer(info["data"], dtype="<u2").copy().reshape(r, c)
        if hashlib.sha256(target.tobytes()).digest() != target_hash:
            raise codec.CodecError("target checksum mismatch")
        result["raw"] = target
        return result
    ctx = codec.contexts(info["reference"], info["labels"], info["flips"], info["thresholds"])
    if fused and planes and _worth_planes(info, ctx, fused_segment):
        return dict(result, **_words_of(info, ctx, stride))
    return _indexed(result, info, ctx, stride, fused, fused_segment)


def _indexed(result, info, ctx, stride, fused, fused_segment):
    """``_read_frame`` from the sections of a frame and the contexts on."""
    r, c = result["shape"]
    n, target_hash = r * c, bytes.fromhex(result["target_sha256"])
    freq = info["main_freq"].reshape(codec.MAIN_CONTEXTS, codec.MAIN_VOCAB)
    seg_len = None
    if fused:
        try:
            seg_len = _fused_segment((r, c), fused_segment)
        except _fused.FusedUnsupported as exc:
            result["fused_reason"] = str(exc)
    # one validated walk serves both indexes when the stride is a multiple of the segment length
    if seg_len and stride % seg_len == 0:
        fs, fo, main = _checkpoints(info["stream"], ctx, freq, codec.MAIN_VOCAB, seg_len)
        states, offsets = fs[::stride // seg_len].copy(), fo[::stride // seg_len].copy()
    else:
        states, offsets, main = _checkpoints(info["stream"], ctx, freq, codec.MAIN_VOCAB, stride)
        if seg_len:
            fs, fo, _ = _checkpoints(info["stream"], ctx, freq, codec.MAIN_VOCAB, seg_len)
    result.update(labels=info["labels"], flips=info["flips"], thresholds=info["thresholds"], main_freq=freq,
                  main_stream=np.frombuffer(info["stream"], dtype=np.uint8).copy(), main_states=states,
                  main_offsets=offsets)
    result["resident_mode"] = info["mode"]
    if seg_len:
        try:
            result["fused_plan"] = _fused.FramePlan((r, c), 16, 16, info["labels"], freq, fs, fo, len(info["stream"]),
                                                    seg_len, image=_word_image, lut_budget=_LUT_BUDGET)
            result["walk_plan"] = result["fused_plan"].for_vector_alus(freq, _WALK_LUT_BUDGET, _word_image)
            result["matrix_plan"] = result["fused_plan"].for_matrix_cores(freq, _MATRIX_LUT_BUDGET, _word_image)
            result["resident_mode"] = 0
        except _fused.FusedUnsupported as exc:
            result["fused_reason"] = str(exc)
    if info["mode"] == 0:
        residual = codec._unpackbits(info["data"], 5, n, "raw5")
        result.update(raw5=np.frombuffer(info["data"], dtype=np.uint8).copy(), residual_symbols=residual)
    else:
        rf = info["residual_freq"].reshape(codec.RES_CONTEXTS, codec.RES_VOCAB)
        rs, ro, residual = _checkpoints(info["residual_stream"], main, rf, codec.RES_VOCAB, stride)
        if result["resident_mode"] == 0:
            # the index builder has decoded and validated the residual stream; it stays on the
            # device as the packed fields the same encoder emits for its mode-0 candidate
            result.update(raw5=np.frombuffer(codec._packbits(residual, 5), dtype=np.uint8).copy())
        else:
            result.update(residual_freq=rf, residual_stream=np.frombuffer(info["residual_stream"], dtype=np.uint8).copy(),
                          residual_states=rs, residual_offsets=ro)
    if hashlib.sha256(codec.join_symbols(main, residual).tobytes()).digest() != target_hash:
        raise codec.CodecError("target checksum mismatch")
    return result


def _worth_planes(info, ctx, fused_segment):
    """Whether the words of a parsed frame are held as planes: not where the fused kernels refuse the frame, nor small matrices
    (``_planes``), nor where the planes would take more than the walk's arrays and 4 %.  What they would list is
    taken from the frame's own frequencies, as each label's words meet them (a row's own eleven exponents are no worse
    on average), so that a frame is decoded once either way."""
    r, c = info["shape"]
    n = r * c
    if n < _planes.FROM_WEIGHTS or c > _planes.MAX_COLS:
        return False
    try:
        seg_len = _fused_segment((r, c), fused_segment)
    except _fused.FusedUnsupported:
        return False
    freq = info["main_freq"].reshape(codec.MAIN_CONTEXTS, codec.MAIN_VOCAB)
    live, sums = (freq > 0).sum(axis=1), freq.sum(axis=1, dtype=np.uint64)
    if not 0 < live.max() <= 255 or not np.isin(sums, (0, 65536)).all():
        return False
    # (a seventh of the words: in all rows, and no multiple of a power of two apart)
    met = np.bincount(ctx.reshape(-1)[::7], minlength=codec.MAIN_CONTEXTS)
    exponents = freq.reshape(16, 16, 2, 256, 4).sum(axis=(2, 4), dtype=np.float64) * met.reshape(16, 16, 1) / 65536
    by_label = exponents.sum(axis=1)
    running = np.concatenate((np.zeros((16, 1)), np.cumsum(by_label, axis=1)), axis=1)
    inside = (running[:, _planes.EXPONENTS:] - running[:, :-_planes.EXPONENTS]).max(axis=1).sum()
    listed = max(0.0, 1 - inside / met.sum()) * n
    # what the arrays of the walk would take: streams, bins, the index and the tables
    walked = len(info["stream"]) + n * 9 // 8 + 8 * r * (c // seg_len + 1) + 16 * (16 * 8 * (int(live.max()) + 1) + _LUT_BUDGET)
    return _planes.plane_bytes(r, c) + 4 * (listed + r + r // 16 * _planes.visits(c)) <= _planes.MEMORY * walked


def _words_of(info, ctx, stride):
    """The words of a frame, validated, with what is needed to make its arrays later (``_indexed``)."""
    r, c = info["shape"]
    freq = info["main_freq"].reshape(codec.MAIN_CONTEXTS, codec.MAIN_VOCAB)
    _, _, main = _checkpoints(info["stream"], ctx, freq, codec.MAIN_VOCAB, stride)
    if info["mode"] == 0:
        residual = codec._unpackbits(info["data"], 5, r * c, "raw5")
    else:
        rf = info["residual_freq"].reshape(codec.RES_CONTEXTS, codec.RES_VOCAB)
        _, _, residual = _checkpoints(info["residual_stream"], main, rf, codec.RES_VOCAB, stride)
    words = codec.join_symbols(main, residual)
    if hashlib.sha256(words.tobytes()).digest() != info["target_sha256"]:
        raise codec.CodecError("target checksum mismatch")
    return dict(words=words.view(np.int16).reshape(r, c), bins=_pairs(ctx), meta=info["meta"], table=info["table"])


def _pairs(ctx):
    """The bins of contexts (their low four bits), two a byte, as the device's plane has them."""
    low = ctx.astype(np.uint8) & 15
    return low[0::2] | low[1::2] << 4


class HipPredictiveTensor:
    """A PPCX-coded BF16 matrix resident on one MI355X; decoding needs the reference matrix."""

    GEMV_UP_TO = 1    # activation rows linear() gives to the vector-ALU kernel
    DENSE_ABOVE = 128  # activation rows above which linear() decodes to a dense transient

    def __init__(self, frame, reference_uint16_numpy, stride=1024, device="cuda:0", *, fused=True,
                 fused_segment=None, resident_contexts=True, m_invariant=False):
        if not isinstance(stride, int) or not 1 <= stride <= 65536:
            raise codec.CodecError("invalid checkpoint stride")
        ix = _read_frame(frame, reference_uint16_numpy, stride, fused=fused, fused_segment=fused_segment, planes=resident_contexts)
        import torch
        if not torch.cuda.is_available():
            raise RuntimeError("a ROCm GPU is required")
        from .bitexact_context_gpu import device_index
        self._lib = _native.hip()
        self.m_invariant = bool(m_invariant)  # linear()'s default for batch_invariant
        self.stride = stride
        self.device = torch.device(device)
        self._index = device_index(self.device)
        self._asked_segment = fused_segment
        self.error = torch.zeros((), device=self.device, dtype=torch.int32)
        if "words" in ix:
            self._hold_planes(ix)
            return
        self._hold_streams(ix)
        # What the tile walker needs of the reference is the 4-bit bin of every word (the
        # decoded word itself comes from the frame's symbols alone), and the reference is given
        # here, once.  Keeping that plane, half a byte per weight, takes the reference out of
        # every later call: a product is then one launch over the frame's bytes and the plane,
        # with no dense reference anywhere.  (The reference's kernels form the bin from the
        # reference word inside the decode loop, GCR/bitexact_predictive_gpu_kernels.py:36-42,
        # which needs the dense reference resident.)
        self.has_contexts = False
        if self.fused is not None and resident_contexts:
            words = np.ascontiguousarray(reference_uint16_numpy, dtype=np.uint16).reshape(self.shape)
            ref = torch.from_numpy(words).to(self.device)  # transient
            with torch.cuda.device(self.device):
                bins, status = self._bins(ref)
                torch.cuda.synchronize(self.device)
            self._status(status, False)
            self.buffers["context_bins"] = bins
            self.has_contexts = True
            del ref

    # As a ``HipContextTensor`` does, one that is held as planes (the words laid out, which needs no contexts and takes less than the
    # frame with them) runs its calls on them for good; the frame's own arrays, plans and descriptors are made when they
    # are asked for and held beside the planes from then on.
    _planes = None
    _WALK = frozenset(("buffers", "fused", "fused_gemm", "fused_matrix", "fused_plan", "_plan", "_matrix_plan", "_walk_plan", "_frame",
                       "_tilings", "_workspace", "_raw5_segment", "_raw5_block", "_rows_held"))

    def __getattr__(self, name):  # (only of what the object does not have)
        held = self.__dict__
        if name in HipPredictiveTensor._WALK and held.get("_planes") is not None:
            from .bitexact_context_gpu import _walk_lock
            with _walk_lock:
                if "buffers" not in held:
                    held.update(self._walk_attributes())  # (all at once: other threads look without the lock)
            if name in held:
                return held[name]
        raise AttributeError(f"{type(self).__name__!r} object has no attribute {name!r}")

    @property
    def fusable(self):
        """Whether products take a kernel of their own (asked without having the walk's arrays made, as ``fused`` has)."""
        return self._planes is not None or self.fused is not None

    def _launch(self, fn, *args):
        from .bitexact_context_gpu import launch_on
        self._status(launch_on(self._index, fn, *args), False)

    def _hold_planes(self, read):
        import torch
        planes = _planes.Planes.of_words(torch.from_numpy(read["words"]).to(self.device), self._launch)
        torch.cuda.current_stream(self.device).synchronize()  # (a first product may be on another stream)
        self.n = math.prod(read["shape"])
        for name in ("shape", "mode", "frame_bytes", "frame_sha256", "source_sha256", "target_sha256", "reference_sha256"):
            setattr(self, name, read[name])
        self.resident_mode, self.fused_reason, self.has_contexts = 0, None, True
        self._kept = {name: read[name] for name in ("bins", "meta", "table")}
        self._planes = planes

    def _walk_attributes(self):
        """The walk's attributes of a tensor that is held as planes: of the words, coded once more with the frame's own frequencies
        in the contexts that were kept of the reference, which gives the same main stream, and packed residuals."""
        import copy
        import torch
        r, c = self.shape
        words = self.decode(None, check=False).view(torch.int16).cpu().numpy().view(np.uint16)
        main, residual = codec.split_symbols(words.reshape(-1))
        meta = codec._inflate(self._kept["meta"], 2 * r + 30)
        labels, flips = (np.frombuffer(meta[i * r:(i + 1) * r], dtype=np.uint8).copy() for i in range(2))
        freq = np.frombuffer(codec._inflate(self._kept["table"], codec.MAIN_CONTEXTS * codec.MAIN_VOCAB * 4), dtype="<u4").copy()
        bins = self._kept["bins"]
        ctx = np.repeat(labels.astype(np.uint16) * 16, c)
        ctx[0::2] += bins & 15
        ctx[1::2] += bins >> 4
        info = dict(mode=0, labels=labels, flips=flips, thresholds=np.frombuffer(meta[2 * r:], dtype="<u2").copy(), main_freq=freq,
                    stream=codec._encode_given(main, ctx, freq), data=codec._packbits(residual, 5))
        about = dict(shape=self.shape, mode=self.mode, target_sha256=self.target_sha256)
        other = copy.copy(self)  # (so that this object has none of them until all are made)
        other._planes = None
        other._hold_streams(_indexed(about, info, ctx, self.stride, True, self._asked_segment))
        if other._raw5_segment:
            bins = _fused.order_records(bins, r, c, other._raw5_segment, other._raw5_block, other.buffers["row_pos"].cpu().numpy(),
                                        other._rows_held, 32, 16)
        other.buffers["context_bins"] = torch.from_numpy(np.ascontiguousarray(bins).view(np.int32)).to(self.device)
        made = {name: value for name, value in vars(other).items() if name in HipPredictiveTensor._WALK}
        return {**made, "fused_reason": other.fused_reason}

    def _hold_streams(self, ix):
        """The device arrays of a frame that is walked where it lies, from what ``_read_frame`` gave."""
        import torch
        self.shape = ix["shape"]
        self.n = math.prod(self.shape)
        self.mode = ix["mode"]
        self.resident_mode = ix.get("resident_mode", self.mode)
        self._plan = ix.pop("fused_plan", None)         # of grouped matrix-core launches ...
        self._matrix_plan = ix.pop("matrix_plan", None)  # ... of the others of these ...
        self._walk_plan = ix.pop("walk_plan", None)     # ... and of one row and the store sink (one plan for most matrices)
        self.fused_reason = ix.pop("fused_reason", None)
        for key in ("source_sha256", "target_sha256", "reference_sha256", "frame_sha256", "frame_bytes"):
            if key in ix:
                setattr(self, key, ix[key])
        buffers = {}
        # The packed residuals -- and the plane of reference bins made below -- in the order the
        # tile walker reads them: records of 32 symbols (20 and 16 bytes), rows by label as the
        # tilings take them, in blocks of as many rows as a wave unit of the GEMV has; inside a
        # block by position in the segment, then by segment, then by row (the order the context
        # codec's tensors give their 12-byte groups, for the same reason: the lanes of a unit then
        # read one run of bytes per visit and a 128-byte line is not visited four times).
        self._raw5_segment = self._raw5_block = self._rows_held = 0
        if self._plan is not None and "raw5" in ix and self.resident_mode == 0:
            block, position, held = self._walk_plan.residual_order()
            rows_, cols_ = self.shape
            ix["raw5"] = _fused.order_records(ix["raw5"], rows_, cols_, self._plan.seg_len, block, position, held, 32, 20)
            ix["row_pos"] = position
            self._raw5_segment, self._raw5_block, self._rows_held = self._plan.seg_len, block, held
        for name, array in ix.items():
            if isinstance(array, np.ndarray) and name != "residual_symbols":
                if name in ("raw5", "main_stream"):  # the kernels read whole dwords / 16-byte chunks at the end
                    array = np.concatenate((array, np.zeros(16, dtype=np.uint8)))
                buffers[name] = torch.from_numpy(np.ascontiguousarray(array)).to(self.device)
        for name in ("main", "residual"):
            if name + "_freq" in ix:
                cum = _tables.cumulative(ix[name + "_freq"])
                buffers[name + "_cum"] = torch.from_numpy(cum).to(self.device)
                buffers[name + "_bucket"] = torch.from_numpy(_tables.coarse_buckets(cum)).to(self.device)
        self._tilings, self._workspace = {}, {}
        self.buffers = buffers
        self._bind()

    def _bind(self):
        """Descriptors over this object's device buffers (their addresses go into the structures
        the kernels take)."""
        self._frame = None
        if self.mode != 2:
            b = self.buffers
            f = _hip_abi.GrfPpcxFrame()
            f.main.bytes, f.main.n_bytes = b["main_stream"].data_ptr(), b["main_stream"].numel() - 16
            f.main.vocab, f.main.nctx = codec.MAIN_VOCAB, codec.MAIN_CONTEXTS
            f.main.cum, f.main.bucket = b["main_cum"].data_ptr(), b["main_bucket"].data_ptr()
            f.main.states, f.main.offsets = b["main_states"].data_ptr(), b["main_offsets"].data_ptr()
            if self.resident_mode == 0:
                f.residual.bytes, f.residual.n_bytes = b["raw5"].data_ptr(), b["raw5"].numel() - 16
                f.raw5_segment, f.raw5_block_rows = self._raw5_segment, self._raw5_block
                f.raw5_row_pos = b["row_pos"].data_ptr() if self._raw5_segment else None
            else:
                f.residual.bytes, f.residual.n_bytes = b["residual_stream"].data_ptr(), b["residual_stream"].numel()
                f.residual.vocab, f.residual.nctx = codec.RES_VOCAB, codec.RES_CONTEXTS
                f.residual.cum, f.residual.bucket = b["residual_cum"].data_ptr(), b["residual_bucket"].data_ptr()
                f.residual.states = b["residual_states"].data_ptr()
                f.residual.offsets = b["residual_offsets"].data_ptr()
            f.labels, f.flips, f.thresholds = b["labels"].data_ptr(), b["flips"].data_ptr(), b["thresholds"].data_ptr()
            f.rows, f.cols = self.shape
            f.mode, f.stride = self.resident_mode, self.stride
            self._frame = f
        self.fused = self.fused_gemm = self.fused_matrix = None
        if self._plan is not None:
            try:
                self._prepare_fused()
            except _fused.FusedUnsupported as exc:
                self.fused, self.fused_reason = None, str(exc)

    def clone(self):
        """A second resident copy of the same coded matrix: every device buffer is duplicated
        (nothing is decoded or indexed again)."""
        import copy
        import torch
        other = copy.copy(self)
        if other._planes is not None:  # (the copy makes its walk's arrays itself, should they be asked for)
            for name in HipPredictiveTensor._WALK:
                vars(other).pop(name, None)
            other.fused_reason = None
            other._planes = other._planes.clone()
            other.error = torch.zeros_like(self.error)
            return other
        other.buffers = {k: v.clone() for k, v in self.buffers.items()}
        other.error = torch.zeros_like(self.error)
        other._tilings, other._workspace = {}, {}
        other._bind()
        return other

    @property
    def resident_bytes(self):
        """Every device allocation this tensor holds: buffers, tilings made so far, the error word."""
        p = self._planes
        total = 4 + (p.nbytes if p is not None else 0)
        if p is not None and "buffers" not in vars(self):
            return total
        total += sum(t.numel() * t.element_size() for t in self.buffers.values())
        total += sum(rows.numel() * 4 + classes.numel() for _, rows, classes, _ in self._tilings.values())
        return int(total)

    @property
    def host_bytes(self):
        """What a tensor that is held as planes keeps in host memory for its walk's arrays, should they be asked for: half a byte a weight, the
        contexts that its words were coded in (the device had them where the frame was walked), and the frame's tables."""
        return sum(len(value) for value in self._kept.values()) if self._planes is not None else 0

    def _prepare_fused(self):
        """Upload the walker's derived arrays: segment index, per-label tables, store tiling."""
        import torch
        plan, b = self._plan, self.buffers
        states, offsets = plan.seg_state, plan.seg_offset
        if self._raw5_segment and "fused_seg_state" not in b:  # the index in the residuals' blocked order
            spr, position = self.shape[1] // self._raw5_segment, b["row_pos"].cpu().numpy()
            states = _fused.order_index(states, self.shape[0], spr, self._raw5_block, position, self._rows_held)
            offsets = _fused.order_index(offsets, self.shape[0], spr, self._raw5_block, position, self._rows_held)
        walk, matrix = self._walk_plan, self._matrix_plan
        arrays = {"fused_seg_state": states, "fused_seg_offset": offsets, "fused_lut": plan.lut, "fused_tab": plan.tab.view(np.int64)}
        if walk is not plan:
            arrays["fused_walk_lut"] = walk.lut
        if matrix is not plan:
            arrays["fused_matrix_lut"] = matrix.lut
        for name, array in arrays.items():
            if name not in b:  # (a clone already holds its copies)
                b[name] = torch.from_numpy(np.ascontiguousarray(array)).to(self.device)

        def frame(of, lut):
            f = _hip_abi.GrfPpcxFused()
            f.main_bytes, f.raw5 = b["main_stream"].data_ptr(), b["raw5"].data_ptr()
            f.seg_state, f.seg_offset = b["fused_seg_state"].data_ptr(), b["fused_seg_offset"].data_ptr()
            f.lut, f.tab = b[lut].data_ptr(), b["fused_tab"].data_ptr()
            f.main_n_bytes = b["main_stream"].numel() - 16
            f.rows, f.cols = self.shape
            f.n_labels = 16
            sc = of.scalars()
            for key in ("seg_len", "segs_per_row", "shift", "lognb", "tabn", "whole_range"):
                setattr(f, key, sc[key])
            f.raw_interleaved = self._raw5_block if self._raw5_segment else 0
            f.row_pos = b["row_pos"].data_ptr() if self._raw5_segment else None
            return f

        self.fused_gemm = frame(plan, "fused_lut")
        self.fused_matrix = self.fused_gemm if matrix is plan else frame(matrix, "fused_matrix_lut")
        self.fused = self.fused_gemm if walk is plan else frame(walk, "fused_walk_lut")
        self.fused_plan = dict(walk.scalars(), **self._tiling_for("waves")[3])

    def index_slot(self, row, segment):
        """Where the checkpoint of ``segment`` (0..segments per row; the last is the end of the
        row's stream) of ``row`` lies in ``buffers["fused_seg_state"]`` / ``["fused_seg_offset"]``
        (blocked order when the residuals are resident in it, else the frame's order)."""
        spr = self.shape[1] // self._plan.seg_len
        if not self._raw5_segment:
            return row * spr + segment
        q, block = int(self.buffers["row_pos"][row].item()), self._raw5_block
        return ((q // block) * (spr + 1) + segment) * block + q % block

    def _tiling_for(self, key):
        """Device copy of a tiling: "waves" = the GEMV and the store sink (wave units, one tiling for
        every row count), "gemm"; of the slab kernels, which only callers of the C entry points
        reach: 0 = store sink, 1/2/4/8 = GEMV row buckets."""
        if key not in self._tilings:
            import torch
            host = (self._matrix_plan.gemm_tiling(self._matrix_plan is self._plan) if key == "gemm" else self._walk_plan.tiling(_fused.WAVE_ROWS_PER_PASS, waves=True)
                    if key == "waves" else self._walk_plan.tiling(key))
            rows = torch.from_numpy(host["tile_rows"].view(np.int32)).to(self.device)
            classes = torch.from_numpy(host["tile_class"]).to(self.device)
            g = _hip_abi.GrfFusedTiling()
            g.tile_rows, g.tile_class = rows.data_ptr(), classes.data_ptr()
            for name, value in host["scalars"].items():
                setattr(g, name, value)
            self._tilings[key] = (g, rows, classes, dict(host["scalars"], lds=host["lds"]))
        return self._tilings[key]

    def _bins(self, ref):
        """Transient plane of 4-bit bins of the reference words (one launch)."""
        import torch
        b = self.buffers
        stream = torch.cuda.current_stream(self.device).cuda_stream
        if self._raw5_segment:  # in the residuals' blocked order (dwords of positions no row has stay unwritten, unread)
            bins = torch.empty(self._rows_held * self.shape[1] // 8, device=self.device, dtype=torch.int32)
            status = self._lib.grf_ppcx_bins_ordered(ref.data_ptr(), b["flips"].data_ptr(), b["thresholds"].data_ptr(),
                                                     self.shape[0], self.shape[1], self._raw5_segment, self._raw5_block,
                                                     b["row_pos"].data_ptr(), bins.data_ptr(), stream)
        else:
            bins = torch.empty(self.n // 8, device=self.device, dtype=torch.int32)
            status = self._lib.grf_ppcx_bins(ref.data_ptr(), b["flips"].data_ptr(), b["thresholds"].data_ptr(),
                                             self.shape[0], self.shape[1], bins.data_ptr(), stream)
        return bins, status

    def _contexts(self, reference_bf16_device):
        """(bins plane, status): the resident plane, or one made from the reference given."""
        if self.has_contexts:
            return self.buffers["context_bins"], 0
        if reference_bf16_device is None:
            raise ValueError("this tensor keeps no context plane: the reference must be given")
        return self._bins(self._reference(reference_bf16_device))

    def _reference(self, reference_bf16_device):
        import torch
        if reference_bf16_device is None:
            raise ValueError("the one-lane-per-checkpoint kernel decodes against the reference: it must be given")
        ref = reference_bf16_device.to(device=self.device).contiguous()
        if tuple(ref.shape) != tuple(self.shape) or ref.dtype != torch.bfloat16:
            raise ValueError("reference device tensor shape/dtype mismatch")
        return ref

    def linear(self, reference_bf16_device, x, bias=None, *, check=False, batch_invariant=None):
        """y = x W^T + bias with W decoded on the fly against the reference: the fused GEMV for
        one activation row, the fused GEMM (matrix cores, one launch) for up to 128; above that
        the fused decode to a dense transient plus a matmul (``dense_linear``), or of planes the product of
        many rows (``planes_prompt``), is faster, unless
        ``batch_invariant`` asks for the fused GEMM throughout, whose rows do not depend on
        the batch.  Frames the tile walker cannot take are decoded and multiplied densely."""
        import torch
        from .bitexact_context_gpu import PackedActivations, dense_linear, planes_prompt
        if isinstance(x, PackedActivations):  # packed for the matrix-core kernel, which is what it gets
            return self._product(reference_bf16_device, x, bias, check, True)
        if batch_invariant is None:  # the tensor's policy
            batch_invariant = self.m_invariant
        m = x.numel() // x.shape[-1] if x.shape[-1] else 0
        if not self.fusable or x.dtype != torch.bfloat16:
            return torch.nn.functional.linear(x, self.decode(reference_bf16_device, check=check), bias)
        if m > self.DENSE_ABOVE and not batch_invariant:
            p = self._planes
            y = planes_prompt(self, p, x, bias) if p is not None else None
            if y is not None:
                return y
            return dense_linear(self._lib, x, self.decode(reference_bf16_device, check=check), bias, self._index)
        return self._product(reference_bf16_device, x, bias, check, batch_invariant or m > self.GEMV_UP_TO)

    def gemv(self, reference_bf16_device, x, bias=None, *, check=False):
        """Fused decode-GEMV (vector ALUs) for 1..8 activation rows; a row's result does not
        depend on how many rows the call carries."""
        if not 1 <= math.prod(x.shape[:-1]) <= 8:
            raise ValueError("gemv takes 1..8 activation rows")
        return self._product(reference_bf16_device, x, bias, check, False)

    def gemm(self, reference_bf16_device, x, bias=None, *, check=False):
        """Fused decode-GEMM (matrix cores) for any number of activation rows, batch-invariant."""
        return self._product(reference_bf16_device, x, bias, check, True)

    def _product(self, reference_bf16_device, x, bias, check, use_gemm):
        import torch
        from .bitexact_context_gpu import PackedActivations, bias_for, launch_on, planes_product, rows_for
        p = self._planes  # (another thread may ask for the arrays)
        if p is not None:
            if not use_gemm and isinstance(x, PackedActivations):
                raise ValueError("packed activations go to the GEMM of a weight of their width on their device")
            return planes_product(self, p, x, bias)
        if self.fused is None:
            raise codec.CodecError("frame is not eligible for the fused kernels: " + str(self.fused_reason))
        packed = x if isinstance(x, PackedActivations) else None
        rows, cols = self.shape
        if packed is not None:
            if not use_gemm or packed.cols != cols or packed.buffer.device != self.device:
                raise ValueError("packed activations go to the GEMM of a weight of their width on their device")
            m, lead, xp, ldx = packed.rows, packed.lead, None, 0
            y = torch.empty((*lead, rows), device=self.device, dtype=torch.bfloat16)
        else:
            if x.dtype is not torch.bfloat16:
                raise ValueError("activation must be bfloat16")
            if x.shape[-1] != cols:
                raise ValueError("activation width does not match the weight")
            x2, ldx = rows_for(x, cols, self._index, self.device)
            m, xp = x2.numel() // cols, x2.data_ptr()
            y = x2.new_empty((*x.shape[:-1], rows))
        bias = bias_for(bias, self._index, self.device)
        if m:
            if check:  # between checks the word keeps what earlier launches reported
                self.error.zero_()
            if self.has_contexts:
                bins, status = self.buffers["context_bins"], 0
            else:
                with torch.cuda.device(self.device):
                    bins, status = self._contexts(reference_bf16_device)
            if not status:
                extra = ()
                if use_gemm:
                    fn, frame, tiling = self._lib.grf_ppcx_gemm, self.fused_matrix, self._tiling_for("gemm")[0]
                    key = m if m <= PackedActivations.MAX_ROWS else PackedActivations.MAX_ROWS
                    size = self._workspace.get((key, tiling.k_parts))
                    if size is None:
                        size = self._lib.grf_gemm_workspace_bytes_split(cols, rows, tiling.k_parts, key)
                        self._workspace[key, tiling.k_parts] = size
                    # transient: the activations in the matrix cores' operand order (+ the parts' sums)
                    space = packed.ensure(size) if packed is not None else x2.new_empty((size + 1) // 2)
                    extra = (space.data_ptr(), size)
                else:
                    fn, frame, tiling = self._lib.grf_ppcx_gemv, self.fused, self._tiling_for("waves")[0]
                status = launch_on(self._index, fn, ctypes.byref(frame), ctypes.byref(tiling), bins.data_ptr(), xp, ldx,
                                   m, y.data_ptr(), rows, bias.data_ptr() if bias is not None else None, *extra,
                                   self.error.data_ptr())
            self._status(status, check)
        return y

    def _raise_launch(self, status):
        self._status(status, False)

    def _status(self, status, check):
        if status:
            raise codec.CodecError(f"device decode launch failed ({status}): "
                                   + self._lib.grf_last_error().decode(errors="replace"))
        if check and self.error.item():
            raise codec.CodecError("HIP PPCX checkpoint/context mismatch")

    def decode(self, reference_bf16_device, check=True, *, general=False):
        """BF16 [rows, cols].  Frames the tile walker supports take two launches (bins of the
        reference, then the walk); ``general`` forces the one-lane-per-checkpoint kernel."""
        import torch
        p = self._planes
        if p is not None and not general:
            out = torch.empty(self.shape, device=self.device, dtype=torch.bfloat16)
            self._launch(self._lib.grf_planes_decode, p.address, out.data_ptr())
            return out
        if self.mode == 2:
            return self.buffers["raw"].view(torch.bfloat16).reshape(self.shape)
        if self.fused is not None and not general:
            out = torch.empty(self.shape, device=self.device, dtype=torch.uint16)
            if check:  # between checks the word keeps what earlier launches reported
                self.error.zero_()
            with torch.cuda.device(self.device):
                bins, status = self._contexts(reference_bf16_device)
                if not status:
                    status = self._lib.grf_ppcx_fused_decode(ctypes.byref(self.fused),
                                                             ctypes.byref(self._tiling_for("waves")[0]), bins.data_ptr(),
                                                             out.data_ptr(), self.error.data_ptr(),
                                                             torch.cuda.current_stream(self.device).cuda_stream)
            self._status(status, check)
            return out.view(torch.bfloat16)
        ref = self._reference(reference_bf16_device)
        count = (self.n + self.stride - 1) // self.stride
        out = torch.empty(count * self.stride, device=self.device, dtype=torch.uint16)
        if check:  # between checks the word keeps what earlier launches reported
            self.error.zero_()
        with torch.cuda.device(self.device):
            status = self._lib.grf_ppcx_decode(ctypes.byref(self._frame), ref.data_ptr(), out.data_ptr(),
                                               self.error.data_ptr(),
                                               torch.cuda.current_stream(self.device).cuda_stream)
        self._status(status, check)
        return out[:self.n].view(torch.bfloat16).reshape(self.shape)


class HipPredictiveGroup:
    """PPCX-coded matrices of one width that take the same activations, multiplied in one launch
    (``grf_ppcx_gemv_group`` / ``grf_ppcx_gemm_group``): what ``HipLinearGroup`` is for tensors
    of the context codec.  The members keep their context planes resident (no reference is
    passed at call time), share one segment length and stay usable on their own; a member's
    rows get the kernel family, and with it the bits, of its own ``linear``."""

    def __init__(self, tensors, *, m_invariant=None):
        import torch
        self.tensors = list(tensors)
        if not 1 <= len(self.tensors) <= 4:
            raise ValueError("a group has 1..4 members")
        first = self.tensors[0]
        for t in self.tensors:
            if not t.fusable:
                raise codec.CodecError("frame is not eligible for the fused kernels: " + str(t.fused_reason))
            if not t.has_contexts:
                raise ValueError("group members keep their context planes resident (resident_contexts=True)")
            if t.shape[1] != first.shape[1] or t.device != first.device:
                raise ValueError("group members need one width and one device")
        self.device, self._lib = first.device, first._lib
        self.m_invariant = any(t.m_invariant for t in self.tensors) if m_invariant is None else bool(m_invariant)
        self.error = torch.zeros((), device=self.device, dtype=torch.int32)
        self._tilings, self._pointer_arrays = {}, {}
        self._index = first._index
        # members whose frames are walked, beside others that are held as planes, have a launch of their own
        self._walked = None  # (their places, their group)
        rest = [i for i, t in enumerate(self.tensors) if t._planes is None]
        if len(rest) == len(self.tensors):
            for key in ("waves", "gemm"):
                self._tiling(key)  # raises FusedUnsupported when the members cannot share a tiling
        elif rest:
            self._walked = rest, HipPredictiveGroup([self.tensors[i] for i in rest], m_invariant=self.m_invariant)
            self._walked[1].error = self.error  # (what a caller polls)

    def _tiling(self, key):
        import torch
        if key not in self._tilings:
            hosts = (_fused.plan_group([t._plan for t in self.tensors], gemm=True) if key == "gemm"
                     else _fused.plan_group([t._walk_plan for t in self.tensors], m=_fused.WAVE_ROWS_PER_PASS, waves=True))
            made = []
            for host in hosts:
                rows = torch.from_numpy(host["tile_rows"].view(np.int32)).to(self.device)
                classes = torch.from_numpy(host["tile_class"]).to(self.device)
                g = _hip_abi.GrfFusedTiling()
                g.tile_rows, g.tile_class = rows.data_ptr(), classes.data_ptr()
                for name, value in host["scalars"].items():
                    setattr(g, name, value)
                made.append((g, rows, classes, dict(host["scalars"], lds=host["lds"])))
            self._tilings[key] = made
        return self._tilings[key]

    def _arrays(self, key, outs, biases):
        n = len(self.tensors)
        if key not in self._pointer_arrays:  # frames, tilings, planes and row counts do not change between calls
            self._pointer_arrays[key] = (
                (ctypes.POINTER(_hip_abi.GrfPpcxFused) * n)(*[ctypes.pointer(t.fused_gemm if key == "gemm" else t.fused)
                                                             for t in self.tensors]),
                (ctypes.POINTER(_hip_abi.GrfFusedTiling) * n)(*[ctypes.pointer(g[0]) for g in self._tiling(key)]),
                (ctypes.c_void_p * n)(*[t.buffers["context_bins"].data_ptr() for t in self.tensors]),
                (ctypes.c_uint32 * n)(*[t.shape[0] for t in self.tensors]), ctypes.c_void_p * n)
        frames, tiles, bins, ldy, pointers = self._pointer_arrays[key]
        ys = pointers(*[y.data_ptr() for y in outs])
        bias = pointers(*[b.data_ptr() if b is not None else None for b in biases])
        return frames, tiles, bins, ys, ldy, bias

    def linear(self, x, biases=None, *, check=False, batch_invariant=None):
        """[x @ W.T (+ bias) for every member]; x is BF16 [..., K] or ``PackedActivations``.
        One activation row goes to the vector-ALU kernel, up to 128 to the matrix cores (every
        row count under ``batch_invariant``), more than that to the members' own ``linear``."""
        import torch
        from .bitexact_context_gpu import PackedActivations, bias_for, launch_on, planes_group, rows_for
        n = len(self.tensors)
        biases = list(biases) if biases is not None else [None] * n
        if len(biases) != n:
            raise ValueError("one bias (or None) per member")
        packed = x if isinstance(x, PackedActivations) else None
        m = packed.rows if packed else math.prod(x.shape[:-1])
        lead = packed.lead if packed else tuple(x.shape[:-1])
        cols = self.tensors[0].shape[1]
        if batch_invariant is None:
            batch_invariant = self.m_invariant
        first = self.tensors[0]
        if packed is None and m > first.DENSE_ABOVE and not batch_invariant:
            return [t.linear(None, x, b, check=check, batch_invariant=False) for t, b in zip(self.tensors, biases)]
        use_gemm = packed is not None or batch_invariant or m > first.GEMV_UP_TO
        planes = [t._planes for t in self.tensors]
        if any(p is not None for p in planes):
            outs = planes_group(self, planes, x, biases)
            if self._walked is not None:
                rest, walked = self._walked
                for i, y in zip(rest, walked.linear(x, [biases[i] for i in rest], check=check, batch_invariant=batch_invariant)):
                    outs[i] = y
            return outs
        if packed is not None:
            if packed.cols != cols or packed.buffer.device != self.device:
                raise ValueError("packed activations of another width or device")
            x2 = None
        else:
            if x.dtype is not torch.bfloat16 or x.shape[-1] != cols:
                raise ValueError("activation must be bfloat16 with the weights' input width")
            x2, ldx = rows_for(x, cols, first._index, self.device)
        biases = [bias_for(b, first._index, self.device) for b in biases]
        outs = [torch.empty((*lead, t.shape[0]), device=self.device, dtype=torch.bfloat16) for t in self.tensors]
        if m:
            if check:
                self.error.zero_()
            xp, ldx = (x2.data_ptr(), ldx) if x2 is not None else (None, 0)
            if use_gemm:
                frames, tiles, bins, ys, ldy, bias = self._arrays("gemm", outs, biases)
                space = packed.buffer if packed else torch.empty(
                    self._lib.grf_gemm_workspace_bytes(cols, m), device=self.device, dtype=torch.uint8)
                status = launch_on(first._index, self._lib.grf_ppcx_gemm_group, n, frames, tiles, bins, xp, ldx, m, ys, ldy,
                                   bias, space.data_ptr(), space.numel(), self.error.data_ptr())
            else:
                frames, tiles, bins, ys, ldy, bias = self._arrays("waves", outs, biases)
                status = launch_on(first._index, self._lib.grf_ppcx_gemv_group, n, frames, tiles, bins, xp, ldx, m, ys, ldy,
                                   bias, self.error.data_ptr())
            if status:
                raise codec.CodecError(f"device launch failed ({status}): "
                                       + self._lib.grf_last_error().decode(errors="replace"))
            if check and self.error.item() != 0:
                raise codec.CodecError("HIP PPCX checkpoint/context mismatch")
        return outs


CudaPredictiveTensor = HipPredictiveTensor
