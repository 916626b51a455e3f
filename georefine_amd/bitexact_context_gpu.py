"""Indexed device decoding of unchanged BCTX frames on MI355X.

``index_frame`` and ``HipContextTensor`` keep the contract of the reference's
``index_frame`` / ``CudaContextTensor`` (GCR/bitexact_context_gpu.py:66-106 and
:109-168): the loader calls ``factory(frame, stride=..., device=...)`` and uses
``shape``, ``source_sha256``, ``frame_sha256``, ``frame_bytes``, ``resident_bytes``,
``decode(check=)`` and ``gather_rows(ids, check=)``.

A frame is validated and decoded on the host when it is loaded, and its matrix is then held in one of two forms.  Most
are laid out as planes (``_planes``: signs and mantissas as they are, exponents two to seven bits), which
take the memory of the frame with its index and go at the memory's pace.  Small matrices and those whose frames are much
smaller than planes stay as frames; of one that is held as planes the frame's arrays are made beside them should they be asked for.  They are the
main stream byte for byte, with a checkpoint index, and the residual section, with one exception: conditional residuals (mode 128) of a frame
that the fused kernels take are kept as packed 6-bit fields, the form mode 0
frames carry (``resident_mode`` 0, ``mode`` 128; ``resident_bytes`` then exceeds the
frame's size by the difference).  Every kernel is hand-written HIP behind the C ABI.
"""
from __future__ import annotations

import ctypes
import hashlib
import math
import os
import threading

import numpy as np

from . import _fused, _hip_abi, _native, _planes, _tables
from . import bitexact_context_codec as base

# The GEMV's tiling scheme: wave units unless the environment asks for the slab kernels.
GEMV_WAVES = os.environ.get("GEOREFINE_FUSED_GEMV", "waves") != "slabs"
WAVE_ROWS = _fused.WAVE_ROWS_PER_PASS


def _ptr(a, ctype):
    return a.ctypes.data_as(ctypes.POINTER(ctype))


def checkpoints(stream, freq, rows, columns, shape, nr, nc, stride, main=None):
    """(states, offsets, symbols) of one stream via ``bcx_checkpoint``."""
    n = math.prod(shape)
    data = np.frombuffer(stream, dtype=np.uint8)
    count = (n + stride - 1) // stride
    states = np.empty(count, dtype=np.uint32)
    offsets = np.empty(count, dtype=np.uint32)
    out = np.empty(n, dtype=np.uint16)
    freq = np.ascontiguousarray(freq, dtype=np.uint32)
    context = _native.U16P() if main is None else _ptr(main, ctypes.c_uint16)
    status = _native.codec().bcx_checkpoint(
        _ptr(data, ctypes.c_uint8) if len(data) else _native.U8P(), len(data), n, shape[0], shape[1],
        _ptr(rows, ctypes.c_uint8), _ptr(columns, ctypes.c_uint8), nr, nc, int(main is not None), context,
        _ptr(freq, ctypes.c_uint32), stride, _ptr(states, ctypes.c_uint32), _ptr(offsets, ctypes.c_uint32),
        _ptr(out, ctypes.c_uint16))
    if status:
        raise base.CodecError(f"checkpoint validation failed ({status})")
    return states, offsets, out


def index_frame(frame: bytes, stride: int = 1024, *, fused_segment=None, raw6_residual=False):
    """Parse, validate and index a frame; the decoded words must hash to the header digest.

    With ``fused_segment`` (a segment length dividing the row length) the result also
    carries ``fused_states`` / ``fused_offsets``, the main-stream index at that length.
    One validated walk serves both indexes when the lengths are multiples of each other.

    ``raw6_residual``: a mode-128 frame's residual section is validated, decoded and
    re-packed into the 6-bit raw form (the form the encoder itself emits for mode 0,
    GCR/bitexact_context_ans.cpp:328-345); the result then carries ``resident_mode`` 0 and
    no residual index.  The main stream's bytes are never altered.

    The arrays are the caller's own: writable, and none of them keeps the frame alive."""
    out = _index_views(frame, stride, fused_segment, raw6_residual)
    for name in ("main_stream", "residual_stream"):
        if name in out:
            out[name] = out[name].copy()
    return out


def _index_views(frame, stride, fused_segment, raw6_residual):
    """``index_frame`` with the two streams as read-only views (of the frame; a re-packed residual
    section: of its own bytes), for a caller that makes arrays of its own from them."""
    return _views_of(*_read_frame(frame, stride, fused_segment, raw6_residual))


def _read_frame(frame, stride, fused_segment, raw6_residual):
    """The validated walk of a frame; what it gives is for ``_views_of``, whose arguments come after it."""
    if not isinstance(stride, int) or not 1 <= stride <= 65536:
        raise base.CodecError("invalid checkpoint stride")
    if len(frame) < base.HEADER.size + 32:
        raise base.CodecError("invalid frame checksum/length")
    mode = base.HEADER.unpack_from(frame)[2]
    repack = raw6_residual and mode == 128
    fine = fused_segment if fused_segment and (mode == 0 or repack) else None
    one_walk = fine is not None and stride % fine == 0  # every stride // fine-th entry of the fine index is the coarse one
    info = base.read_words(frame, fine if one_walk else stride, "checkpoint validation failed ({})".format)
    if mode != 1 and info["words_digest"] != info["digest"]:
        raise base.CodecError("indexed source checksum mismatch")
    return info, len(frame), stride, fine, repack


def _views_of(info, frame_bytes, stride, fine, repack):
    r, c = info["shape"]
    mode, one_walk = info["mode"], fine is not None and stride % fine == 0
    out = {"shape": (r, c), "mode": mode, "nr": info["nr"], "nc": info["nc"], "stride": stride,
           "source_sha256": info["digest"].hex(), "frame_sha256": info["frame_sha256"], "frame_bytes": frame_bytes}
    if mode == 1:
        out["raw"] = info["raw"].reshape(-1).astype(np.uint16)
        out["resident_mode"] = 1
        return out
    rows, columns, sf = info["rows"], info["columns"], info["main_freq"]
    out["resident_mode"] = 0 if repack else mode
    states, offsets = info["main_states"], info["main_offsets"]
    if one_walk:
        out.update(fused_states=states, fused_offsets=offsets, fused_segment=fine)
        states, offsets = states[::stride // fine].copy(), offsets[::stride // fine].copy()
    elif fine:
        fs, fo, _ = checkpoints(info["main_stream"], sf, rows, columns, (r, c), info["nr"], info["nc"], fine)
        out.update(fused_states=fs, fused_offsets=fo, fused_segment=fine)
    residual = info["residual_stream"]
    if repack:
        residual = base._pack6(base._lib(), info["words"])
    elif mode == 128:
        main = (info["words"] >> 5) & np.uint16(0x3FF)
        rf = info["residual_freq"]
        out.update(zip(("residual_freq", "residual_states", "residual_offsets"),
                       (rf, *checkpoints(residual, rf, rows, columns, (r, c), info["nr"], info["nc"], stride, main)[:2])))
    out.update(rows=rows, columns=columns, main_freq=sf, main_stream=np.frombuffer(info["main_stream"], dtype=np.uint8),
               main_states=states, main_offsets=offsets, residual_stream=np.frombuffer(residual, dtype=np.uint8))
    return out


def _device_stream(buffers, name, stream, vocab, nctx):
    s = _hip_abi.GrfStream()
    s.bytes = buffers[stream].data_ptr()
    s.n_bytes = buffers[stream].numel()
    s.vocab, s.nctx = vocab, nctx
    if name + "_cum" in buffers:
        s.cum = buffers[name + "_cum"].data_ptr()
        s.bucket = buffers[name + "_bucket"].data_ptr()
        s.states = buffers[name + "_states"].data_ptr()
        s.offsets = buffers[name + "_offsets"].data_ptr()
    return s


GEMV_UP_TO = 2             # activation rows linear() gives to the vector-ALU kernel
GEMM_TWO_ROWS_FROM = 8192  # row length from which two activation rows go to the matrix-core kernel
DENSE_ABOVE = 128          # activation rows above which linear() decodes to a dense transient

# Words of pinned host memory that launches report to and their callers read after a wait; a call
# takes one and gives it back zeroed, at most this many stay.
_host_words = []
HOST_WORDS_KEPT = 16


def _host_word():
    """One of the kept words, or a new one.  (Asked for by taking it: between a look at the list and
    the taking another thread may take the last.)"""
    try:
        return _host_words.pop()
    except IndexError:
        import torch
        return torch.zeros(1, dtype=torch.int32, pin_memory=True)


# Counters of gathers under way, by device; a call takes some and gives them back, as it does a word.
_done_counters = {}
# Words and counters of calls that were left before their launch was known to be over: it may write them yet, so they are
# held for as long as the program runs and nothing else is put in their place.
_left_behind = []


def _counters_for(index):
    try:
        return _done_counters.setdefault(index, []).pop()
    except IndexError:
        import torch
        return torch.zeros(_hip_abi.GATHER_COUNTER_BYTES // 4, dtype=torch.int32, device=f"cuda:{index}")


# How long a gather is polled for before the thread sleeps until the stream is done.
GATHER_SPIN_US = 100


def gather_polled(count, waves):
    """Whether a lookup of ``count`` rows, each a workgroup of ``waves``, tells the host that it is over and is polled for: while all of
    them find a place on the GPU at once (256 units of 28 waves), and not of more rows than come on at a few a unit.  Where they follow one
    another, what a workgroup's end waits for costs more than a wait for the stream (``GatherDone`` has the measurements)."""
    return count < 4000 and count * waves <= 7168


def route_rows(m, cols, invariant=False):
    """The kernel family that takes ``m`` activation rows of a matrix with ``cols`` columns:
    ``"gemv"`` (vector ALUs), ``"gemm"`` (matrix cores) or ``"dense"`` (fused decode + library
    matmul).  One rule for single matrices and grouped launches.

    ``invariant``: every row count takes the matrix-core kernel, whose accumulation order per
    output element is fixed by the matrix alone -- row m of an M-row call then has the bits of
    the one-row call (the property GS/miv_gemv.py:1-9 states for M <= 8 and
    GS/bi_csrc/bi_gemm.cuh:1-17 for any M: a speculative verify pass at M = k + 1 reproduces the
    decode steps).  Without it the fastest family per row count is chosen: the GEMV for one
    row and for two rows of a short-row matrix (its second row costs 44 % at K = 17408, where
    its activations no longer stay in the first-level cache), the GEMM to 128 rows, the dense
    route above; rows are then bit-equal only between calls that take the same family."""
    if invariant:
        return "gemm"
    if m > DENSE_ABOVE:
        return "dense"
    if m == 0 or m > GEMV_UP_TO or (m == 2 and cols >= GEMM_TWO_ROWS_FROM):
        return "gemm"
    return "gemv"


def device_index(device):
    """The ordinal of a torch device ("cuda" alone: the current one)."""
    import torch
    return device.index if device.index is not None else torch.cuda.current_device()


def launch_on(index, fn, *args):
    """``fn(*args, stream)`` with GPU ``index`` current, on its current stream.  (The handle as
    torch's own generated code takes it, and the device switched only when it is another one: the
    stream object and the context manager cost more than the launch.)"""
    import torch
    if torch._C._cuda_getDevice() == index:
        return fn(*args, torch._C._cuda_getCurrentRawStream(index))
    with torch.cuda.device(index):
        return fn(*args, torch._C._cuda_getCurrentRawStream(index))


def rows_for(x, cols, index, device):
    """``x`` as rows of ``cols`` BF16 values the kernels can read where they are (16-byte aligned,
    rows a multiple of 8 apart); the common case, a contiguous tensor on the device, as it is."""
    if x.get_device() == index and x.is_contiguous() and not x.data_ptr() & 15:
        return x, cols
    x2 = x.reshape(-1, cols).to(device)
    if x2.stride(-1) != 1 or x2.stride(0) % 8 or x2.data_ptr() & 15:
        import torch
        x2 = x2.clone(memory_format=torch.contiguous_format)
    return x2, x2.stride(0)


def bias_for(bias, index, device):
    """A bias vector as the kernels take it (BF16, contiguous, on the device)."""
    import torch
    if bias is None or (bias.dtype is torch.bfloat16 and bias.get_device() == index and bias.is_contiguous()):
        return bias
    return bias.to(device=device, dtype=torch.bfloat16).contiguous()


def _plain(t, index):
    """A BF16 tensor on the GPU that is nothing but its values: no subclass, no zeros without memory, no gradient asked for."""
    import torch
    return (type(t) in (torch.Tensor, torch.nn.Parameter) and t.dtype is torch.bfloat16 and t.get_device() == index and t.layout is torch.strided
            and not t.is_neg() and not t._is_zerotensor() and not (t.requires_grad and torch.is_grad_enabled()))


def _observed():
    """Whether torch would do more with an operator than run it: a transform, a mode, a tracer, autocast."""
    import torch
    return (torch.is_autocast_enabled("cuda") or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
            or torch._C._functorch.peek_interpreter_stack() is not None or torch._C._get_tracing_state() is not None
            or torch.autograd.forward_ad._current_level >= 0)


def _only_values(x, bias, rows, cols, index):
    """Whether a product of many rows is asked for nothing but its values, in a form that torch would take."""
    return (_plain(x, index) and x.dim() and x.shape[-1] == cols
            and (bias is None or _plain(bias, index) and bias.shape == (rows,) and bias.is_contiguous()) and not _observed())


def _prompt_rows(x, cols, index):
    import torch
    x2, ldx = rows_for(x, cols, index, x.device)
    if not cols <= ldx <= 1 << 21:  # (rows that overlap, or lie too far apart)
        return x2.clone(memory_format=torch.contiguous_format), cols
    return x2, ldx


def planes_prompt(tensor, p, x, bias):
    """The product of many rows with the planes ``p`` as they are, or None where the decoded matrix is the faster
    way (``grf_planes_prompt_plan``) or more than the values is asked for, as in ``dense_linear``."""
    rows, cols = tensor.shape
    lib, index, m = tensor._lib, tensor._index, x.numel() // cols
    plan = lib.grf_planes_prompt_plan(rows, cols, m) if m < 1 << 30 else -1
    if plan < 0 or not _only_values(x, bias, rows, cols, index):
        return None
    x2, ldx = _prompt_rows(x, cols, index)
    y = x2.new_empty((*x.shape[:-1], rows))
    size = lib.grf_planes_prompt_workspace_bytes(rows, m, plan)
    space = x2.new_empty(size // 2) if size else None
    status = launch_on(index, lib.grf_planes_prompt, p.address, x2.data_ptr(), ldx, m, plan, y.data_ptr(), rows,
                       bias.data_ptr() if bias is not None else None, space.data_ptr() if size else None, size)
    if status:
        tensor._raise_launch(status)
    return y


def dense_linear(lib, x, weight, bias, index):
    """``F.linear`` of activations with a decoded matrix on GPU ``index``: the library's product, or the one of
    ``grf_dense_gemm`` where that is the faster (its plan says so by the sizes) and nothing but the values
    is asked for.  What torch would refuse, differentiate, trace or convert goes to torch."""
    import torch
    rows, cols = weight.shape
    m = x.numel() // cols if cols else 0
    size = lib.grf_dense_gemm_plan(rows, cols, m) if m < 1 << 30 else -1  # (first: the calls that it sends on pay nothing else)
    if size < 0 or not _only_values(x, bias, rows, cols, index) or not weight.is_contiguous() or weight.data_ptr() & 15:
        return torch.nn.functional.linear(x, weight, bias)
    x2, ldx = _prompt_rows(x, cols, index)
    y = x2.new_empty((*x.shape[:-1], rows))
    space = x2.new_empty(size // 2) if size else None
    status = launch_on(index, lib.grf_dense_gemm, weight.data_ptr(), rows, cols, x2.data_ptr(), ldx, m, y.data_ptr(), rows,
                       bias.data_ptr() if bias is not None else None, space.data_ptr() if size else None, size)
    if status:
        raise base.CodecError(f"device launch failed ({status}): " + lib.grf_last_error().decode(errors="replace"))
    return y


class PackedActivations:
    """Activation rows copied once into the operand order of the matrix-core kernels, for
    several coded matrices that take the same input (q/k/v, gate/up): ``gemm`` and
    ``linear`` of the device tensors accept it in place of ``x``.  At most 128 rows."""

    MAX_ROWS = 128

    def __init__(self, x):
        import torch
        if x.dtype != torch.bfloat16 or not x.is_cuda:
            raise ValueError("activations must be bfloat16 on the device")
        self.lead, self.cols = tuple(x.shape[:-1]), x.shape[-1]
        x2 = x.reshape(-1, self.cols)
        self.rows = x2.shape[0]
        if not 1 <= self.rows <= self.MAX_ROWS or self.cols % 16:
            raise ValueError("1..128 rows of a width that is a multiple of 16")
        if x2.stride(-1) != 1 or x2.stride(0) % 4 or x2.data_ptr() % 8:
            x2 = x2.clone(memory_format=torch.contiguous_format)
        lib = _native.hip()
        size = lib.grf_gemm_workspace_bytes(self.cols, self.rows)
        self.buffer = torch.empty(size, device=x.device, dtype=torch.uint8)
        with torch.cuda.device(x.device):
            status = lib.grf_pack_activations(x2.data_ptr(), x2.stride(0), self.rows, self.cols, self.buffer.data_ptr(),
                                              size, torch.cuda.current_stream(x.device).cuda_stream)
        if status:
            raise base.CodecError(f"device launch failed ({status}): " + lib.grf_last_error().decode(errors="replace"))

    def ensure(self, nbytes):
        """Room behind the packed rows for a consumer whose launch is cut along K (its parts'
        sums live in the same workspace): a larger buffer with the packed rows copied over."""
        import torch
        if self.buffer.numel() < nbytes:
            larger = torch.empty(nbytes, device=self.buffer.device, dtype=torch.uint8)
            larger[:self.buffer.numel()] = self.buffer
            self.buffer = larger
        return self.buffer


class _Buffers(dict):
    """A tensor's device arrays by name.  A tensor that keeps its residual groups in pair form (``residual_pairs``,
    ``GRF_RAW_PAIRS``) lists that array, and answers for ``residual_stream`` as well: the same groups as packed
    fields, made when first asked for and held from then on, so that its address stays good.  The kernels read the pairs;
    an array of packed fields that is put here under the name is what they read after ``_bind``."""

    _packed = (None, None)  # (the pairs it was made of, the packed fields)

    def __missing__(self, name):
        if name != "residual_stream" or "residual_pairs" not in self:
            raise KeyError(name)
        import torch
        pairs = self["residual_pairs"]
        with _packed_lock:
            if self._packed[0] is not pairs:
                packed = _residual_form(pairs.clone(), False)
                torch.cuda.current_stream(pairs.device).synchronize()  # (it may be read on another stream)
                self._packed = pairs, packed
            return self._packed[1]

    def __contains__(self, name):
        return super().__contains__(name) or name == "residual_stream" and super().__contains__("residual_pairs")

    def get(self, name, default=None):
        return self[name] if name in self else default

    def holds(self, name):
        """Whether the array itself is here."""
        return super().__contains__(name)


_packed_lock = threading.Lock()
_walk_lock = threading.RLock()  # (what makes a tensor's walk attributes reads attributes of it)


def _residual_form(groups, to_pairs):
    """12-byte residual groups on the device turned to pair form, or back to packed fields, where they are."""
    import torch
    lib = _native.hip()
    with torch.cuda.device(groups.device):
        status = lib.grf_pair_residuals(groups.data_ptr(), groups.numel(), int(to_pairs),
                                        torch.cuda.current_stream(groups.device).cuda_stream)
    if status:
        raise base.CodecError(f"device launch failed ({status}): " + lib.grf_last_error().decode(errors="replace"))
    return groups


def _stream_arrays(read, fused, residual_block):
    """The arrays of a frame that is walked where it lies, from what ``_read_frame`` gave."""
    indexed = _views_of(*read)
    plan, reason = None, "disabled" if not fused else "frame mode or geometry"
    if "fused_states" in indexed:
        try:
            plan = _fused.FramePlan(indexed["shape"], indexed["nr"], indexed["nc"], indexed["rows"],
                                    indexed["main_freq"], indexed.pop("fused_states"), indexed.pop("fused_offsets"),
                                    len(indexed["main_stream"]), indexed["fused_segment"])
        except _fused.FusedUnsupported as exc:
            reason = str(exc)
            indexed.pop("fused_states", None)
            indexed.pop("fused_offsets", None)
    main_bytes = len(indexed["main_stream"]) if "main_stream" in indexed else 0
    raw6_segment = raw6_block = 0
    if plan is not None:  # the fused kernels read 16-byte vectors: pad the stream's allocation
        indexed["main_stream"] = np.concatenate((indexed["main_stream"], np.zeros(16, dtype=np.uint8)))
        # The packed residuals in the order the tile walker reads them (a permutation of the
        # 12-byte groups of 16 fields, no field is touched): rows by class as the tilings take
        # them, in blocks of as many rows as a wave unit of the GEMV has; inside a block by
        # position in the segment, then by segment, then by row.  The lanes of a unit walk
        # neighbouring segments of the block's rows in step, so they read one run of bytes per
        # visit and a 128-byte line is used in a single visit; in the frame's order a line came
        # back from memory about twice per launch.
        rows_, cols_ = indexed["shape"]
        seg = indexed["fused_segment"]
        raw = indexed["residual_stream"]
        if raw.size == rows_ * cols_ * 3 // 4:
            block, position, held = plan.residual_order(residual_block)
            indexed["residual_stream"] = _fused.order_residuals(raw, rows_, cols_, seg, block, position, held)
            indexed["row_pos"] = position
            raw6_segment, raw6_block = seg, block
        states, offsets = plan.seg_state, plan.seg_offset
        if raw6_segment:  # the segment index in the same blocked order (``_fused.order_index``)
            spr_ = cols_ // seg
            states = _fused.order_index(states, rows_, spr_, block, position, held)
            offsets = _fused.order_index(offsets, rows_, spr_, block, position, held)
        indexed.update(fused_seg_state=states, fused_seg_offset=offsets, fused_lut=plan.lut, fused_tab=plan.tab)
    for name in ("main_stream", "residual_stream"):  # what is still a view: callers may keep the result for long
        if name in indexed and not indexed[name].flags.writeable:
            indexed[name] = indexed[name].copy()
    return {"indexed": indexed, "plan": plan, "reason": reason, "main_bytes": main_bytes, "raw6_segment": raw6_segment,
            "raw6_block": raw6_block}


class _Prepared(dict):
    """What ``HipContextTensor.host_prepare`` gives for a matrix that is held as planes: its words, and what the frame says of
    itself.  The arrays of the walk (``_stream_arrays``) are made when they are asked for."""

    def __init__(self, read, asked, **fields):
        super().__init__(asked, **fields)
        self._read = read

    def __missing__(self, name):
        if name not in ("indexed", "plan", "reason", "main_bytes", "raw6_segment", "raw6_block"):
            raise KeyError(name)
        self.update(_stream_arrays(self._read, True, self["block"]))
        return self[name]

    def __reduce__(self):  # (the streams are views of the frame)
        info = {k: bytes(v) if isinstance(v, memoryview) else v for k, v in self._read[0].items()}
        return _Prepared, ((info, *self._read[1:]), dict(self))


def planes_product(tensor, p, x, bias):
    """A product of a tensor that is held as the planes ``p``, of any number of rows; a row's bits depend on neither
    the batch nor the call.  (Nothing is walked, so there is no checkpoint to miss.)"""
    import torch
    rows, cols = tensor.shape
    packed = isinstance(x, PackedActivations)
    if packed:
        if x.cols != cols or x.buffer.device != tensor.device:
            raise ValueError("packed activations of another width or device")
        lead, m, ldx, x2 = x.lead, x.rows, cols, x.buffer
        y = tensor.error.new_empty((*lead, rows), dtype=torch.bfloat16)
    else:
        if x.dtype is not torch.bfloat16 or x.shape[-1] != cols:
            raise ValueError("activation must be bfloat16 with the weight's input width")
        x2, ldx = rows_for(x, cols, tensor._index, tensor.device)
        if not cols <= ldx <= 1 << 24:  # (rows that overlap, or lie too far apart)
            x2, ldx = x2.reshape(-1, cols).clone(memory_format=torch.contiguous_format), cols
        m = x2.numel() // cols
        y = x2.new_empty((*x.shape[:-1], rows))
    if m:
        bias = bias_for(bias, tensor._index, tensor.device)
        size = p.workspace(m)
        space = tensor.error.new_empty(size // 4) if size else None
        status = launch_on(tensor._index, tensor._lib.grf_planes_linear, p.address, x2.data_ptr(), ldx, m, packed, y.data_ptr(),
                           bias.data_ptr() if bias is not None else None, space.data_ptr() if size else None, size)
        if status:
            tensor._raise_launch(status)
    return y


def planes_group(owner, planes, x, biases):
    """The products of members that are held as ``planes`` (None: another launch's), in one launch: [y or None].  ``owner``
    is the group."""
    import torch
    n, outs = len(planes), [None] * len(planes)
    held = [i for i in range(n) if planes[i] is not None]
    cols, packed = planes[held[0]].cols, isinstance(x, PackedActivations)
    if packed:
        if x.cols != cols or x.buffer.device != owner.device:
            raise ValueError("packed activations of another width or device")
        x2, ldx, m, lead = x.buffer, cols, x.rows, x.lead
    else:
        if x.dtype is not torch.bfloat16 or x.shape[-1] != cols:
            raise ValueError("activation must be bfloat16 with the weights' input width")
        m, lead = math.prod(x.shape[:-1]), tuple(x.shape[:-1])
        x2, ldx = rows_for(x, cols, owner._index, owner.device)
        if not cols <= ldx <= 1 << 24:  # (rows that overlap, or lie too far apart)
            x2, ldx = x2.reshape(-1, cols).clone(memory_format=torch.contiguous_format), cols
    for i in held:
        outs[i] = owner.error.new_empty((*lead, planes[i].rows), dtype=torch.bfloat16)
    if m:
        count = len(held)
        biases = [bias_for(biases[i], owner._index, owner.device) for i in held] if biases is not None else None
        addresses = [planes[i].address for i in held]
        kept = owner._pointer_arrays.get("planes")
        if kept is None or kept[0] != addresses:
            kept = owner._pointer_arrays["planes"] = (
                addresses, (ctypes.c_void_p * count)(*addresses), (ctypes.c_uint32 * count)(*[planes[i].rows for i in held]), ctypes.c_void_p * count)
        _, members, ldy, pointers = kept
        size = sum(planes[i].workspace(m) for i in held) if m > _planes.OWN_ROWS else 0
        space = owner.error.new_empty(size // 4) if size else None
        status = launch_on(owner._index, owner._lib.grf_planes_group, count, members, x2.data_ptr(), ldx, m, packed,
                           pointers(*[outs[i].data_ptr() for i in held]), ldy,
                           pointers(*[b.data_ptr() if b is not None else None for b in biases]) if biases is not None else None,
                           space.data_ptr() if size else None, size)
        if status:
            raise base.CodecError(f"device launch failed ({status}): " + owner._lib.grf_last_error().decode(errors="replace"))
    return outs


class HipContextTensor:
    """A BCTX-coded BF16 matrix resident on one MI355X."""

    GEMV_UP_TO, GEMM_TWO_ROWS_FROM, DENSE_ABOVE = GEMV_UP_TO, GEMM_TWO_ROWS_FROM, DENSE_ABOVE

    @staticmethod
    def host_prepare(frame: bytes, *, stride: int = 1024, fused=True, fused_segment=None, residual_block=None):
        """The host half of the constructor -- parse, validate and index the frame, lay out the
        fused kernels' tables -- for callers that prepare frames on worker threads and construct
        the device objects later (``HipContextTensor(frame, prepared=...)`` then only uploads).
        Needs no GPU."""
        segment = None
        if fused:
            try:
                header = base.HEADER.unpack_from(frame)
                segment = _fused.choose_segment(header[6], fused_segment, rows=header[5])
            except _fused.FusedUnsupported:
                segment = None
        read = _read_frame(frame, stride, segment, segment is not None)
        info = read[0]
        could = segment is not None and GEMV_WAVES and _planes.possible(info)
        sections = None
        if could:  # the frame's labels and tables, as it has them
            meta, tables = base.HEADER.unpack_from(frame)[7:9]
            at = base.HEADER.size
            sections = bytes(frame[at:at + meta]), bytes(frame[at + meta:at + meta + tables])
        asked = {"stride": stride, "fused": fused, "asked_segment": fused_segment, "sections": sections, "block": residual_block}
        if not could or not _planes.worth(info, segment):
            return {**asked, **_stream_arrays(read, fused, residual_block)}
        if residual_block not in (None, 1, 2, 4, 8, 16):
            raise _fused.FusedUnsupported("residual blocks have 1, 2, 4, 8 or 16 rows")
        return _Prepared(read, asked, words=info["words"], shape=info["shape"], mode=info["mode"], nr=info["nr"], nc=info["nc"],
                         source_sha256=info["digest"].hex(), frame_sha256=info["frame_sha256"], frame_bytes=len(frame))

    def __init__(self, frame: bytes, *, stride: int = 1024, device="cuda:0", fused=True, fused_segment=None,
                 m_invariant=False, prepared=None, residual_block=None):
        import torch
        if not torch.cuda.is_available():
            raise RuntimeError("a ROCm GPU is required")
        self._lib = _native.hip()  # fails loudly when the device library is absent
        # linear()'s default routing: True sends every row count to the matrix-core kernel, so
        # that a row's output bits never depend on the rows it arrives with (route_rows)
        self.m_invariant = bool(m_invariant)
        if prepared is None:
            prepared = self.host_prepare(frame, stride=stride, fused=fused, fused_segment=fused_segment,
                                         residual_block=residual_block)
        elif prepared["stride"] != stride or prepared["fused"] != fused:
            raise ValueError("the frame was prepared with another stride or fused setting")
        self.stride = stride
        self.asked_segment = prepared["asked_segment"]  # None: the length was left to ``choose_segment``
        self.device = torch.device(device)
        self._index = device_index(self.device)
        self._error_open = True  # the error word may hold what an unchecked launch reported
        self.error = torch.zeros((), device=self.device, dtype=torch.int32)
        about = prepared if isinstance(prepared, _Prepared) else prepared["indexed"]
        self.shape = about["shape"]
        self.n = math.prod(self.shape)
        self.mode, self.nr, self.nc = about["mode"], about["nr"], about["nc"]
        self.source_sha256 = about["source_sha256"]
        self.frame_sha256 = about["frame_sha256"]
        self.frame_bytes = about["frame_bytes"]
        self._sections, self._block = prepared["sections"], prepared["block"]
        if isinstance(prepared, _Prepared):
            self.resident_mode = 0  # (as the walk would hold it, should it be asked for)
            self.fused_reason = ""
            words = torch.from_numpy(prepared["words"].view(np.int16)).to(self.device).view(self.shape)
            self._hold_planes(words)
        else:
            # form of the residual section on the device: 0 = packed 6-bit, 128 = rANS stream
            self.resident_mode = about["resident_mode"]
            self._hold_streams(prepared)

    # A tensor that is held as planes (``_planes``) runs its products, decode and lookups on them for good.  The frame's own
    # arrays, which the walk of its states takes, their plan and descriptors are made when they are asked for, for the C interface, the
    # one-lane decode or to be looked at, and are held beside the planes from then on: what a call runs, and with it a
    # product's bits, never depends on what was looked at.  Frames that the planes do not take have nothing but those arrays.
    _planes = None
    _WALK = frozenset(("buffers", "fused", "fused_plan", "_plan", "_frame", "_tilings", "_workspace", "_gather", "_main_bytes",
                       "_raw6_segment", "_raw6_block", "_gather_waves"))

    def __getattr__(self, name):  # (only of what the object does not have)
        held = self.__dict__
        if name in HipContextTensor._WALK and held.get("_planes") is not None:
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

    def _hold_planes(self, words):
        import torch
        planes = _planes.Planes.of_words(words, self._launch)
        torch.cuda.current_stream(self.device).synchronize()  # (a first product may be on another stream)
        self.resident_bytes = planes.nbytes + self.error.numel() * self.error.element_size()
        self._planes = planes

    def _walk_attributes(self):
        """The walk's attributes of a tensor that is held as planes: of the words, coded once more with the frame's own labels
        and frequencies, which gives the same main stream, and packed residuals, the form that the walk takes."""
        import copy
        import zlib
        import torch
        words = self.decode(check=False).view(torch.int16).cpu().numpy().view(np.uint16)
        meta, tables = self._sections
        labels = base._inflate_exact(meta, sum(self.shape))
        rows, columns = (np.frombuffer(part, dtype=np.uint8) for part in (labels[:self.shape[0]], labels[self.shape[0]:]))
        frequencies = zlib.decompress(tables)[:self.nr * self.nc * base.MAIN_VOCAB * 4]
        lib = base._lib()
        main = base._encode_stream(lib, words, rows, columns, self.nr, self.nc, 0, frequencies)
        frame = base._sealed(base._sections(0, self.nr, self.nc, *self.shape, meta, zlib.compress(frequencies, 1), main, base._pack6(lib, words),
                                            b"", bytes.fromhex(self.source_sha256)))
        segment = _fused.choose_segment(self.shape[1], self.asked_segment, rows=self.shape[0])
        other = copy.copy(self)  # (so that this object has none of them until all are made)
        other._planes = None
        other._hold_streams(_stream_arrays(_read_frame(frame, self.stride, segment, True), True, self._block))
        other._plan_gather()
        made = {name: value for name, value in vars(other).items() if name in HipContextTensor._WALK}
        beside = self._planes.nbytes  # (the error word is counted with the arrays)
        return {**made, "fused_reason": other.fused_reason, "resident_bytes": other.resident_bytes + beside}

    def _hold_streams(self, prepared):
        """The device arrays of a frame that is walked where it lies."""
        import torch
        indexed, plan = prepared["indexed"], prepared["plan"]
        self._gather = None  # (lanes, piece capacity) of the row gather once planned; False: not possible
        self.fused = None
        self.fused_reason = prepared["reason"]
        self._main_bytes = prepared["main_bytes"]
        self._raw6_segment, self._raw6_block = prepared["raw6_segment"], prepared["raw6_block"]
        buffers = _Buffers()
        for name, array in indexed.items():
            if isinstance(array, np.ndarray):
                buffers[name] = torch.from_numpy(np.ascontiguousarray(array)).to(self.device)
        for name in ("main", "residual"):
            if name + "_freq" in indexed:
                cum = _tables.cumulative(indexed[name + "_freq"])
                buffers[name + "_cum"] = torch.from_numpy(cum).to(self.device)
                buffers[name + "_bucket"] = torch.from_numpy(_tables.coarse_buckets(cum)).to(self.device)
        if self._raw6_segment and GEMV_WAVES:  # (the slab kernels' read-ahead is for packed fields)
            buffers["residual_pairs"] = _residual_form(buffers.pop("residual_stream"), True)
            torch.cuda.current_stream(self.device).synchronize()  # (a first product may be on another stream)
        self.buffers = buffers
        self.resident_bytes = int(sum(t.numel() * t.element_size() for t in self.buffers.values())
                                  + self.error.numel() * self.error.element_size())
        self._plan = plan
        self._bind()

    def _bind(self):
        """Descriptors over this object's device buffers (their addresses go into the structures
        the kernels take), and the first tilings."""
        plan = self._plan
        self._frame = None
        # (an array of packed fields that a caller put in the pairs' place goes first)
        raw = "residual_pairs" if set(self.buffers) & {"residual_pairs", "residual_stream"} == {"residual_pairs"} else "residual_stream"
        form = _hip_abi.RAW_PAIRS if raw == "residual_pairs" else 0
        if self.mode != 1:
            f = _hip_abi.GrfBctxFrame()
            f.main = _device_stream(self.buffers, "main", "main_stream", 1024, self.nr * self.nc)
            f.residual = _device_stream(self.buffers, "residual", raw, 64, 1024)
            f.row_class = self.buffers["rows"].data_ptr()
            f.col_class = self.buffers["columns"].data_ptr()
            f.rows, f.cols = self.shape
            f.nc, f.mode, f.stride = self.nc, self.resident_mode, self.stride
            f.raw6_segment, f.raw6_block_rows = self._raw6_segment, self._raw6_block | form
            f.raw6_row_pos = self.buffers["row_pos"].data_ptr() if self._raw6_segment else None
            f.main.n_bytes = self._main_bytes
            self._frame = f
        self._tilings = {}
        self._workspace = {}  # bytes by (activation rows, parts along K)
        self._gather = None  # (lanes, piece capacity) of the row gather once planned; False: not possible
        if plan is not None:
            d = _hip_abi.GrfBctxFused()
            b = self.buffers
            d.main_bytes, d.raw6 = b["main_stream"].data_ptr(), b[raw].data_ptr()
            d.seg_state, d.seg_offset = b["fused_seg_state"].data_ptr(), b["fused_seg_offset"].data_ptr()
            d.lut, d.tab, d.col_class = b["fused_lut"].data_ptr(), b["fused_tab"].data_ptr(), b["columns"].data_ptr()
            d.main_n_bytes = self._main_bytes
            d.raw_interleaved = self._raw6_block if self._raw6_segment else 0
            d.row_pos = b["row_pos"].data_ptr() if self._raw6_segment else None
            for key, value in plan.scalars().items():
                setattr(d, key, value)
            d.nc |= form
            self.fused = d
            self.fused_plan = plan.scalars()
            self.fused_reason = ""
            try:
                self._tiling(1)
                self._store_tiling()
            except _fused.FusedUnsupported as exc:
                self.fused, self.fused_reason = None, str(exc)
                return
            # the tilings linear() uses are uploaded now, so that a first call launches and
            # nothing else (it may be part of a graph capture)
            try:
                self._tiling(2)
                self._gemm_tiling()
            except _fused.FusedUnsupported:
                pass  # reported by the call that needs it

    def clone(self, residual_block=None):
        """A second resident copy of the same coded matrix: every device buffer is duplicated
        (nothing is decoded or indexed again), so a stack of layers with equal weights can be
        laid out in device memory at the cost of one device-to-device copy each.
        ``residual_block``: the copy keeps its packed residuals in blocks of that many rows (1,
        2, 4, 8 or 16; see ``host_prepare``), re-ordered on the device: a permutation of the
        12-byte groups, no field is touched."""
        import copy
        import torch
        other = copy.copy(self)
        if other._planes is not None:  # (the copy makes its walk's arrays itself, should they be asked for)
            if residual_block is not None:
                if residual_block not in (1, 2, 4, 8, 16):
                    raise ValueError("residual blocks have 1, 2, 4, 8 or 16 rows")
                other._block = residual_block
            for name in HipContextTensor._WALK:
                vars(other).pop(name, None)
            other.fused_reason = ""
            other._planes = other._planes.clone()
            other.error = torch.zeros_like(self.error)
            other.resident_bytes = other._planes.nbytes + other.error.numel() * other.error.element_size()
            return other
        other.buffers = _Buffers((k, v.clone()) for k, v in self.buffers.items())
        if residual_block is not None and self._raw6_segment and residual_block != self._raw6_block:
            if residual_block not in (1, 2, 4, 8, 16):
                raise ValueError("residual blocks have 1, 2, 4, 8 or 16 rows")
            old, groups, spr = self._raw6_block, self._raw6_segment // 16, self.shape[1] // self._raw6_segment
            kept = "residual_stream" if other.buffers.holds("residual_stream") else "residual_pairs"
            raw = other.buffers[kept]
            held = raw.numel() // (groups * spr * 12)  # a multiple of 16: every class starts on one
            by_row = raw[:held * groups * spr * 12].view(held // old, groups, spr, old, 12).permute(0, 3, 1, 2, 4)
            by_row = by_row.reshape(held // residual_block, residual_block, groups, spr, 12)
            other.buffers[kept] = by_row.permute(0, 2, 3, 1, 4).contiguous().view(-1)
            for name in ("fused_seg_state", "fused_seg_offset"):  # the index is in the same blocked order
                kind = other.buffers[name].dtype
                index = other.buffers[name].view(torch.int32).view(held // old, spr + 1, old).permute(0, 2, 1)
                index = index.reshape(held // residual_block, residual_block, spr + 1).permute(0, 2, 1)
                other.buffers[name] = index.contiguous().view(-1).view(kind)
            other._raw6_block = residual_block
        other.error = torch.zeros_like(self.error)
        other.resident_bytes = int(sum(t.numel() * t.element_size() for t in other.buffers.values())
                                   + other.error.numel() * other.error.element_size())
        other._bind()
        return other

    def index_slot(self, row, segment):
        """Where the checkpoint of ``segment`` (0..segments per row; the last is the end of the
        row's stream) of ``row`` lies in ``buffers["fused_seg_state"]`` / ``["fused_seg_offset"]``:
        in the blocked order of the resident residuals when the tensor keeps them so
        (``_fused.order_index``), else in the frame's order."""
        spr = self.shape[1] // self.fused_plan["seg_len"]
        if not self._raw6_segment:
            return row * spr + segment
        q, block = int(self.buffers["row_pos"][row].item()), self._raw6_block
        return ((q // block) * (spr + 1) + segment) * block + q % block

    def _tiling(self, m):
        """Device copy of the tiling used for m activation rows (0 = store sink).  The GEMV has
        one wave-unit tiling for every row count; under GEOREFINE_FUSED_GEMV=slabs (experiments
        and tests of the slab kernels) tilings are made for m in {1, 2, 4, 8} and shared by
        the row counts in between."""
        if m and GEMV_WAVES and "waves" in self._tilings:
            return self._tilings["waves"]
        if m == 0:
            bucket = 0
        elif GEMV_WAVES:
            bucket = "waves"
        else:
            bucket = next(v for v in (1, 2, 4, 8) if v >= m)
        if bucket not in self._tilings:
            self._upload_tiling(bucket, self._plan.tiling(WAVE_ROWS if bucket == "waves" else bucket, waves=bucket == "waves"))
        return self._tilings[bucket]

    def _upload_tiling(self, bucket, host):
        import torch
        rows = torch.from_numpy(host["tile_rows"]).to(self.device)
        classes = torch.from_numpy(host["tile_class"]).to(self.device)
        g = _hip_abi.GrfFusedTiling()
        g.tile_rows, g.tile_class = rows.data_ptr(), classes.data_ptr()
        for key, value in host["scalars"].items():
            setattr(g, key, value)
        self._tilings[bucket] = (g, rows, classes, dict(host["scalars"], lds=host["lds"]))
        self.resident_bytes += rows.numel() * 4 + classes.numel()

    def _store_tiling(self):
        """The tiling decode() uses: wave units of the kernel that stores whole lines where the segments
        allow it, else the GEMV's; the slab tiling of the store sink only with the slab GEMV."""
        if not GEMV_WAVES:
            return self._tiling(0)
        if "lines" not in self._tilings:
            host = self._plan.lines_tiling()
            if host is None:
                return self._tiling(1)
            self._upload_tiling("lines", host)
        return self._tilings["lines"]

    # ------------------------------------------------------------------ decode
    def _decode_blocks(self, blocks=None, *, check=True):
        import torch
        if blocks is None:
            count = (self.n + self.stride - 1) // self.stride
            ids = None
        else:
            blocks = blocks.to(device=self.device, dtype=torch.int64).contiguous().reshape(-1)
            count = blocks.numel()
            ids = blocks.data_ptr()
        result = torch.empty(count * self.stride, device=self.device, dtype=torch.uint16)
        if check:  # between checks the word keeps what earlier launches reported
            self.error.zero_()
        self._error_open = True
        status = launch_on(self._index, self._lib.grf_bctx_decode, ctypes.byref(self._frame), ids, count, result.data_ptr(),
                           self.error.data_ptr())
        if status:
            raise base.CodecError(f"device decode launch failed ({status}): "
                                  + self._lib.grf_last_error().decode(errors="replace"))
        if check and self.error.item() != 0:
            raise base.CodecError("HIP decoder checkpoint mismatch")
        return result.view(torch.bfloat16)

    def _launch(self, fn, *args):
        status = launch_on(self._index, fn, *args)
        if status:
            self._raise_launch(status)

    def _raise_launch(self, status):
        raise base.CodecError(f"device launch failed ({status}): " + self._lib.grf_last_error().decode(errors="replace"))

    def _check(self, check):
        if check and self.error.item() != 0:
            raise base.CodecError("HIP decoder checkpoint mismatch")

    def decode(self, *, check=True, general=False):
        """Dense BF16 matrix.  Fused frames use the store sink of the fused walker;
        ``general=True`` forces the one-lane-per-segment kernel."""
        import torch
        p = self._planes  # (another thread may ask for the arrays)
        if p is not None and not general:
            out = torch.empty(self.shape, device=self.device, dtype=torch.bfloat16)
            self._launch(self._lib.grf_planes_decode, p.address, out.data_ptr())
            return out
        if self.mode == 1:
            return self.buffers["raw"].view(torch.bfloat16).reshape(self.shape)
        if self.fused is None or general:
            return self._decode_blocks(check=check)[:self.n].reshape(self.shape)
        out = torch.empty(self.shape, device=self.device, dtype=torch.bfloat16)
        if check:  # between checks the word keeps what earlier launches reported
            self.error.zero_()
        self._error_open = True
        self._launch(self._lib.grf_bctx_fused_decode, ctypes.byref(self.fused), ctypes.byref(self._store_tiling()[0]),
                     out.data_ptr(), self.error.data_ptr())
        self._check(check)
        return out

    def _gemm_tiling(self):
        if "gemm" not in self._tilings:
            import torch
            host = self._plan.gemm_tiling()
            rows = torch.from_numpy(host["tile_rows"]).to(self.device)
            classes = torch.from_numpy(host["tile_class"]).to(self.device)
            g = _hip_abi.GrfFusedTiling()
            g.tile_rows, g.tile_class = rows.data_ptr(), classes.data_ptr()
            for key, value in host["scalars"].items():
                setattr(g, key, value)
            self._tilings["gemm"] = (g, rows, classes, dict(host["scalars"], lds=host["lds"]))
            self.resident_bytes += rows.numel() * 4 + classes.numel()
        return self._tilings["gemm"]

    def _packed_call(self, packed, bias, check):
        """The GEMM on rows that were packed before (x == NULL in the C call)."""
        import torch
        if packed.cols != self.shape[1] or packed.buffer.device != self.device:
            raise ValueError("packed activations of another width or device")
        bias = bias_for(bias, self._index, self.device)
        y = torch.empty((packed.rows, self.shape[0]), device=self.device, dtype=torch.bfloat16)
        if check:  # between checks the word keeps what earlier launches reported
            self.error.zero_()
        self._error_open = True
        tiling = self._gemm_tiling()[0]
        space = packed.ensure(self._lib.grf_gemm_workspace_bytes_split(self.shape[1], self.shape[0], tiling.k_parts,
                                                                       packed.rows))
        self._launch(self._lib.grf_bctx_gemm, ctypes.byref(self.fused), ctypes.byref(tiling), None, 0,
                     packed.rows, y.data_ptr(), y.stride(0), bias.data_ptr() if bias is not None else None,
                     space.data_ptr(), space.numel(), self.error.data_ptr())
        self._check(check)
        return y.reshape(*packed.lead, self.shape[0])

    def _fused_call(self, fn, tiling, x, bias, check, *, workspace=False):
        import torch
        rows, cols = self.shape
        if x.dtype is not torch.bfloat16 or x.shape[-1] != cols:
            raise ValueError("activation must be bfloat16 with the weight's input width")
        x2, ldx = rows_for(x, cols, self._index, self.device)
        bias = bias_for(bias, self._index, self.device)
        m = x2.numel() // cols
        y = x2.new_empty((*x.shape[:-1], rows))
        if m:
            if check:  # between checks the word keeps what earlier launches reported
                self.error.zero_()
            self._error_open = True
            extra = ()
            if workspace:  # transient: the activations in the matrix cores' operand order (+ the parts' sums)
                key = m if m <= PackedActivations.MAX_ROWS else PackedActivations.MAX_ROWS
                size = self._workspace.get((key, tiling.k_parts))
                if size is None:
                    size = self._lib.grf_gemm_workspace_bytes_split(cols, rows, tiling.k_parts, key)
                    self._workspace[key, tiling.k_parts] = size
                packed = x2.new_empty((size + 1) // 2)
                extra = (packed.data_ptr(), size)
            status = launch_on(self._index, fn, ctypes.byref(self.fused), ctypes.byref(tiling), x2.data_ptr(), ldx, m,
                               y.data_ptr(), rows, bias.data_ptr() if bias is not None else None, *extra,
                               self.error.data_ptr())
            if status:
                self._raise_launch(status)
            if check:
                self._check(check)
        return y

    def gemv(self, x, bias=None, *, check=False):
        """Fused decode-GEMV (vector ALUs) for 1..8 activation rows; the result of a row does
        not depend on how many rows the call carries."""
        p = self._planes
        if p is not None:
            if not 1 <= (x.numel() // x.shape[-1] if x.shape[-1] else 0) <= 8:
                raise ValueError("gemv takes 1..8 activation rows")
            return planes_product(self, p, x, bias)
        if self.fused is None:
            raise base.CodecError("frame is not eligible for the fused kernels: " + self.fused_reason)
        m = x.numel() // x.shape[-1] if x.shape[-1] else 0
        if not 1 <= m <= 8:
            raise ValueError("gemv takes 1..8 activation rows")
        return self._fused_call(self._lib.grf_bctx_gemv, self._tiling(m)[0], x, bias, check)

    def gemm(self, x, bias=None, *, check=False):
        """Fused decode-GEMM (matrix cores) for any number of activation rows, batch-invariant:
        a row's output bits are the same whatever else is in the batch."""
        p = self._planes
        if p is not None:
            return planes_product(self, p, x, bias)
        if self.fused is None:
            raise base.CodecError("frame is not eligible for the fused kernels: " + self.fused_reason)
        if isinstance(x, PackedActivations):
            return self._packed_call(x, bias, check)
        return self._fused_call(self._lib.grf_bctx_gemm, self._gemm_tiling()[0], x, bias, check, workspace=True)

    def linear(self, x, bias=None, *, check=False, batch_invariant=None):
        """y = x @ W.T (+ bias) with W decoded inside the kernel; x is BF16 [..., K].

        The row count picks the kernel family (``route_rows``): by default the fastest one --
        the fused decode-GEMV for one row (and two rows of a short-row matrix), the fused
        decode-GEMM to 128 rows (one launch), above that a fused decode to a dense transient
        and a matmul (``dense_linear``; a second GEMM launch would decode the matrix again), or of planes
        the product of many rows where that is the faster (``planes_prompt``).
        ``batch_invariant=True`` -- or the tensor's ``m_invariant`` policy, which is the default
        when the argument is left out -- sends every row count through the GEMM, so that a
        row's output never depends on the batch it arrives in: ``linear(x[:1])`` is
        ``linear(x[:6])[:1]`` bit for bit.  Frames the fused kernels cannot take are decoded on
        the device and multiplied densely.  ``check=True`` reads the error word back (a host
        sync)."""
        if isinstance(x, PackedActivations):  # packed for the matrix-core kernel, which is what it gets
            return self.gemm(x, bias, check=check)
        if batch_invariant is None:
            batch_invariant = self.m_invariant
        width = x.shape[-1]
        m = x.numel() // width if width else math.prod(x.shape[:-1])
        p = self._planes
        held = p is not None
        if held and (m <= DENSE_ABOVE or batch_invariant):
            return planes_product(self, p, x, bias)
        route = "dense" if held or self.fused is None else route_rows(m, self.shape[1], batch_invariant)
        if route == "dense":
            import torch
            x = x.to(self.device)
            y = planes_prompt(self, p, x, bias) if held else None
            if y is not None:
                return y
            weight = self.decode(check=check)
            if not held and self.fused is None:  # any number of rows, and another decode (or none) than the product's plan counts on
                return torch.nn.functional.linear(x, weight, bias)
            return dense_linear(self._lib, x, weight, bias, self._index)
        if route == "gemm":
            return self.gemm(x, bias, check=check)
        return self.gemv(x, bias, check=check)

    def gather_rows(self, ids, *, check=True, validate=True):
        """Rows ``ids`` (any shape) as BF16 [*ids.shape, cols]; IndexError for a row the matrix
        does not have (GCR/bitexact_context_gpu.py:159-168).  Frames the tile walker takes give
        every requested row a workgroup that walks all of its segments at once; others decode
        the checkpoint blocks of the rows, one lane each.  ``validate=False`` (with
        ``check=False``) leaves out the range test, which reads a flag back from the device, for
        callers that vouch for their ids and must not synchronise (a HIP graph capture); ids
        outside the matrix are then clamped into it."""
        import torch
        if ids.dtype is not torch.int64 or ids.get_device() != self._index:
            ids = ids.to(device=self.device, dtype=torch.int64)
        if ids.numel() == 0:
            return torch.empty((*ids.shape, self.shape[1]), device=self.device, dtype=torch.bfloat16)
        p = self._planes
        if p is not None:
            return self._gather_planes(p, ids, validate)
        self._plan_gather()
        if self.fused is not None and self._gather:
            return self._gather_fused(ids, check, validate)
        if validate:
            if torch.any((ids < 0) | (ids >= self.shape[0])).item():
                raise IndexError("embedding row outside tensor")
        else:
            ids = ids.clamp(0, self.shape[0] - 1)
        if self.mode == 1 or self.shape[1] % self.stride:
            return self.decode(check=check)[ids]
        per_row = self.shape[1] // self.stride
        blocks = (ids.reshape(-1, 1) * per_row + torch.arange(per_row, device=self.device)).reshape(-1)
        return self._decode_blocks(blocks, check=check).reshape(*ids.shape, self.shape[1])

    def _plan_gather(self):
        if self.fused is not None and self._gather is None:
            try:
                shape = self._plan.gather_shape()
                self._gather_waves = min(16, -(-self.fused.segs_per_row // shape[0]))
                self._gather = shape  # (last: another thread goes by it)
            except _fused.FusedUnsupported:
                self._gather = False

    def _gather_fused(self, ids, check, validate):
        """One launch, which also looks up classes and tests the ids; what it finds wrong it writes to a word of
        pinned host memory, which nothing has to copy back, and, unless there are many rows (``gather_polled``), that it is
        over to the same word, which is polled.  A caller that waits for the stream next, with nothing launched between, waits 6 us
        for the runtime to ask for a signal then (us, 777 rows of 8192 x 5120: lookup and wait 40.6, with the wait for the stream in the
        lookup 34.4; lookups one after the other 29.3 and 31.4, two launches on the rows and then a wait 50.5 and 53.0).  An event
        recorded while the rows are under way makes the first 34.6 and every lookup 0.3 to 1.2 longer, so there is none."""
        import torch
        ids = ids.contiguous()
        out = torch.empty((*ids.shape, self.shape[1]), device=self.device, dtype=torch.bfloat16)
        if check and self._error_open:  # between checks the word keeps what earlier launches reported
            self.error.zero_()
            self._error_open = False
        elif not check:
            self._error_open = True
        about = (ctypes.byref(self.fused), *self._gather, self.buffers["rows"].data_ptr(), ids.data_ptr(), ids.numel(), out.data_ptr())
        if not (check or validate):
            self._launch(self._lib.grf_bctx_gather_rows, *about, self.error.data_ptr(), None)
            return out

        def launch(where, counters):
            report = where if check else self.error.data_ptr(), where if validate else None
            if counters is not None:
                self._launch(self._lib.grf_bctx_gather_rows_done, *about, *report, counters.data_ptr(), where)
            else:
                self._launch(self._lib.grf_bctx_gather_rows, *about, *report)

        found = self._told(launch, gather_polled(ids.numel(), self._gather_waves))
        if found & _hip_abi.ERR_INDEX:
            raise IndexError("embedding row outside tensor")
        if found:
            self.error.fill_(found)
            self._error_open = True
            raise base.CodecError("HIP decoder checkpoint mismatch")
        return out

    def _told(self, launch, polled):
        """What a lookup reports, once it is over: ``launch(address of the word, counters or None)`` starts it."""
        import torch
        word, counters = _host_word(), _counters_for(self._index) if polled else None
        where = word.data_ptr()
        try:
            launch(where, counters)
            found = self._lib.grf_take_word(where, _hip_abi.GATHER_DONE, GATHER_SPIN_US) if polled else 0
            if not found:
                torch.cuda.current_stream(self._index).synchronize()
                value = ctypes.c_int32.from_address(where)  # (a tensor's element costs twice the time)
                found, value.value = value.value, 0
        except BaseException:
            _left_behind.append((word, counters))
            raise
        if len(_host_words) < HOST_WORDS_KEPT:
            _host_words.append(word)
        if polled and len(_done_counters[self._index]) < HOST_WORDS_KEPT:
            _done_counters[self._index].append(counters)
        return found & ~_hip_abi.GATHER_DONE

    def _gather_planes(self, p, ids, validate):
        """Of a tensor that is held as planes: one launch, of whose findings only refused ids are left to wait for."""
        import torch
        ids = ids.contiguous()
        out = torch.empty((*ids.shape, self.shape[1]), device=self.device, dtype=torch.bfloat16)
        about = p.address, ids.data_ptr(), ids.numel(), out.data_ptr()
        launch = lambda where, counters: self._launch(self._lib.grf_planes_gather, *about, where,
                                                      counters.data_ptr() if counters is not None else None,
                                                      where if counters is not None else None)
        if not validate:
            launch(None, None)
        elif self._told(launch, gather_polled(ids.numel(), -(-_planes.visits(self.shape[1]) // 16))):
            raise IndexError("embedding row outside tensor")
        return out


class HipLinearGroup:
    """Coded matrices of one width that take the same activations (q/k/v, gate/up), multiplied
    in one launch: the members' tiles share the grid, so a small matrix fills the workgroup
    slots a large one leaves, and the launch overhead is paid once.  The members stay usable
    on their own.  Members whose index was left to the default go together whatever lengths their
    sizes gave them; lengths that were asked for (``HipContextTensor(..., fused_segment=...)``)
    must be one."""

    def __init__(self, tensors, *, m_invariant=None):
        import torch
        self.tensors = list(tensors)
        if not 1 <= len(self.tensors) <= 4:
            raise ValueError("a group has 1..4 members")
        first = self.tensors[0]
        for t in self.tensors:
            if not t.fusable:
                raise base.CodecError("frame is not eligible for the fused kernels: " + t.fused_reason)
            if t.shape[1] != first.shape[1] or t.device != first.device:
                raise ValueError("group members need one width and one device")
        if len({t.asked_segment for t in self.tensors} - {None}) > 1:
            raise _fused.FusedUnsupported("group members were asked to have different segment lengths")
        self.device, self._lib, self._index = first.device, first._lib, first._index
        # the members' policy unless given: a group of members that keep rows bit-equal across
        # row counts does so too
        self.m_invariant = any(t.m_invariant for t in self.tensors) if m_invariant is None else bool(m_invariant)
        self.error = torch.zeros((), device=self.device, dtype=torch.int32)
        self._tilings, self._pointer_arrays, self._workspace = {}, {}, {}
        # Members whose frames are walked, beside others that are held as planes, have a launch of their own: laid out for the planes' launch
        # they would lose the bits of their own products, which the vector-ALU route gives every member.  (Small matrices are walked: one row of
        # 2048 and 256 x 1024 takes 15.8 us in two launches, where one of planes would take 4.4.)
        self._walked = None  # (their places, their group)
        rest = [i for i, t in enumerate(self.tensors) if t._planes is None]
        if len(rest) == len(self.tensors):
            self._plan_tilings()
        elif rest:
            self._walked = rest, HipLinearGroup([self.tensors[i] for i in rest], m_invariant=self.m_invariant)
            self._walked[1].error = self.error  # (what a caller polls)

    def _plan_tilings(self):
        for key in (1, 2, "gemm"):
            self._tiling(key)  # raises FusedUnsupported when the members cannot share a tiling

    def _tiling(self, key):
        """Per member: (structure, device arrays) of the joint tiling for ``key`` (GEMV row
        bucket 1/2/4/8, or "gemm")."""
        import torch
        if key not in self._tilings:
            plans = [t._plan for t in self.tensors]
            hosts = (_fused.plan_group(plans, gemm=True, mixed=True) if key == "gemm"
                     else _fused.plan_group(plans, m=key, waves=GEMV_WAVES, mixed=True))
            made = []
            for host in hosts:
                rows = torch.from_numpy(host["tile_rows"]).to(self.device)
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
        if key not in self._pointer_arrays:  # frames, tilings and row counts do not change between calls
            tilings = self._tiling(key)
            self._pointer_arrays[key] = (
                (ctypes.POINTER(_hip_abi.GrfBctxFused) * n)(*[ctypes.pointer(t.fused) for t in self.tensors]),
                (ctypes.POINTER(_hip_abi.GrfFusedTiling) * n)(*[ctypes.pointer(g[0]) for g in tilings]),
                (ctypes.c_uint32 * n)(*[t.shape[0] for t in self.tensors]), ctypes.c_void_p * n)
        frames, tiles, ldy, pointers = self._pointer_arrays[key]
        ys = pointers(*[y.data_ptr() for y in outs])
        bias = pointers(*[b.data_ptr() if b is not None else None for b in biases]) if biases else None
        return frames, tiles, ys, ldy, bias

    def linear(self, x, biases=None, *, check=False, batch_invariant=None):
        """[x @ W.T (+ bias) for every member]; x is BF16 [..., K] or ``PackedActivations``.
        Row counts are routed by the rule of ``HipContextTensor.linear`` (``route_rows``), so a
        member gets the kernel family, and with it the bits, of its own ``linear``; above 128
        rows the members' own decode + matmul."""
        import torch
        n = len(self.tensors)
        if biases is not None:
            biases = list(biases)
            if len(biases) != n:
                raise ValueError("one bias (or None) per member")
            if not any(b is not None for b in biases):
                biases = None
        cols = self.tensors[0].shape[1]
        packed = x if isinstance(x, PackedActivations) else None
        if packed is not None:
            m, lead = packed.rows, packed.lead
        else:
            lead, width = x.shape[:-1], x.shape[-1]
            m = x.numel() // width if width else math.prod(lead)
        if batch_invariant is None:
            batch_invariant = self.m_invariant
        route = "gemm" if packed is not None else route_rows(m, cols, batch_invariant)
        if route == "dense":
            return [t.linear(x, b, check=check, batch_invariant=False)
                    for t, b in zip(self.tensors, biases if biases is not None else [None] * n)]
        planes = [t._planes for t in self.tensors]
        if any(p is not None for p in planes):
            return self._linear_planes(planes, x, biases, check, batch_invariant)
        if packed is not None:
            if packed.cols != cols or packed.buffer.device != self.device:
                raise ValueError("packed activations of another width or device")
            x2, xp, ldx, make = None, None, 0, self.error.new_empty
        else:
            if x.dtype is not torch.bfloat16 or width != cols:
                raise ValueError("activation must be bfloat16 with the weights' input width")
            x2, ldx = rows_for(x, cols, self._index, self.device)
            xp, make = x2.data_ptr(), x2.new_empty
        if biases is not None:
            biases = [bias_for(b, self._index, self.device) for b in biases]
        outs = [make((*lead, t.shape[0]), dtype=torch.bfloat16) for t in self.tensors]
        if m:
            if check:
                self.error.zero_()
            if route == "gemm":
                frames, tiles, ys, ldy, bias = self._arrays("gemm", outs, biases)
                if packed is not None:
                    space, size = packed.buffer, packed.buffer.numel()
                else:
                    key = m if m <= PackedActivations.MAX_ROWS else PackedActivations.MAX_ROWS
                    size = self._workspace.get(key)
                    if size is None:
                        size = self._workspace[key] = self._lib.grf_gemm_workspace_bytes(cols, key)
                    space = x2.new_empty((size + 1) // 2)
                status = launch_on(self._index, self._lib.grf_bctx_gemm_group, n, frames, tiles, xp, ldx, m, ys, ldy, bias,
                                   space.data_ptr(), size, self.error.data_ptr())
            else:
                frames, tiles, ys, ldy, bias = self._arrays(next(v for v in (1, 2, 4, 8) if v >= m), outs, biases)
                status = launch_on(self._index, self._lib.grf_bctx_gemv_group, n, frames, tiles, xp, ldx, m, ys, ldy, bias,
                                   self.error.data_ptr())
            if status:
                raise base.CodecError(f"device launch failed ({status}): "
                                      + self._lib.grf_last_error().decode(errors="replace"))
            if check and self.error.item() != 0:
                raise base.CodecError("HIP decoder checkpoint mismatch")
        return outs


    def _linear_planes(self, planes, x, biases, check, batch_invariant):
        """Up to 128 rows of a group some of whose members are held as planes: one launch for those, and one for the rest."""
        outs = planes_group(self, planes, x, biases)
        if self._walked is not None:
            rest, walked = self._walked
            for i, y in zip(rest, walked.linear(x, [biases[i] for i in rest] if biases is not None else None, check=check,
                                                batch_invariant=batch_invariant)):
                outs[i] = y
        return outs


# The loaders name the class they expect; keep that name importable.
CudaContextTensor = HipContextTensor
