"""Matrices resident as planes: which ones, how a product's sums are split, and the device arrays.

The planes (``csrc/word_planes.h``, ``csrc/planes.hip``) hold a matrix's words at fixed places in 11.5 bits a weight and a
list of the few whose exponent is outside the eleven that hold most of their row.  A context frame with
the index its walk needs takes as much (5120 x 17408 of normal weights with a scale a row: 11.6 bits either way;
small matrices, whose index is finer and whose tables do not shrink, 13 to 30), and its walk is bound by the vector ALUs where the planes are
read at the memory's pace.  us, walk / planes: one row of 17408 x 5120 twice 110 / 51, six of 5120 x 17408 69 / 36, 64 of the
first 151 / 73, a decode of 5120 x 6144 39 / 25, 777 of 8192 rows looked up 16 / 7.
"""
from __future__ import annotations

import ctypes

import numpy as np

from . import _hip_abi, _native

VISIT, UNIT, VISIT_BYTES, UNIT_BYTES = 256, 64, 5888, 1536  # csrc/word_planes.h
EXPONENTS = 11
MAX_COLS = 1 << 17
OWN_ROWS = 8  # activation rows up to which a launch needs no workspace (a matrix alone is given one where it pays)
# Weights from which a matrix is laid out.  Smaller ones have shorter kernels as planes too for up to 32 rows and for more than 128 (us of
# launches in a row, walked and as planes: 256 x 512 one row 6.6 3.8, 32 rows 6.9 4.5, 200 13.5 11.4; 511 x 1024 8.1 4.1, 9.3 4.9, 15.7 14.0; a call
# by itself 9.0 8.0), but longer ones between (64 and 128 rows of 256 x 512 8.0 10.2, 11.1 13.9; of 300 x 1744 10.8 13.5, 14.5 19.1; of
# 511 x 1024 12.4 10.9, 13.7 14.9).
FROM_WEIGHTS = 1 << 19
# How much more memory than the frame's arrays the planes may take (frames of few exponents code far below 11.5 bits
# and stay frames).
MEMORY = 1.04


def visits(cols):
    """Visits of 256 columns, the last one of up to three units of 64."""
    return cols // VISIT + (cols % VISIT > 0)


def plane_bytes(rows, cols):
    units = (cols % VISIT + UNIT - 1) // UNIT
    return -(-rows // 16) * (cols // VISIT * VISIT_BYTES + units * UNIT_BYTES)


def listed_share(row_class, col_class, main_freq, nr, nc):
    """The share of words that the planes would list, by the frame's own frequencies: outside the best eleven
    exponents of each row class (a row's own are no worse on average)."""
    exponents = np.asarray(main_freq, dtype=np.float64).reshape(nr, nc, 256, 4).sum(axis=3) / 65536
    by_row = np.einsum("rce,c->re", exponents, np.bincount(col_class, minlength=nc) / len(col_class))
    running = np.concatenate((np.zeros((nr, 1)), np.cumsum(by_row, axis=1)), axis=1)
    inside = (running[:, EXPONENTS:] - running[:, :-EXPONENTS]).max(axis=1)
    return float((1 - inside) @ np.bincount(row_class, minlength=nr) / len(row_class))


def possible(info):
    """Whether the matrix of a parsed context frame (``bitexact_context_codec.read_words``) can be held as planes."""
    rows, cols = info["shape"]
    if info["mode"] not in (0, 128) or cols > MAX_COLS or cols % 16 or rows * cols > 0xFFFFFFFF:
        return False
    return 0 < int((info["main_freq"] > 0).sum(axis=1).max()) <= 255  # (what the fused kernels refuse stays refused)


def worth(info, segment):
    """Whether it is, where the walk would index it at ``segment``: from ``FROM_WEIGHTS`` on, where the planes take no more memory
    than the frame's arrays and 4 %."""
    rows, cols = info["shape"]
    n, nr, nc = rows * cols, info["nr"], info["nc"]
    if n < FROM_WEIGHTS:
        return False
    live = int((info["main_freq"] > 0).sum(axis=1).max())
    tables = nr * nc * 9 * 1024 + nr * (nc * 8 * (live + 1) + 32768)
    frame = len(info["main_stream"]) + n * 3 // 4 + 8 * rows * (cols // segment + 1) + tables
    listed = listed_share(info["rows"], info["columns"], info["main_freq"], nr, nc) * n
    return plane_bytes(rows, cols) + 4 * (listed + rows + rows // 16 * visits(cols)) <= MEMORY * frame


def sum_splits(rows, cols):
    """Splits of a product's sums (``grf_planes``), by the matrix's sizes alone.  A batch's workgroups, eight row blocks of one split
    each, are dealt to 256 compute units: the busiest one's visits count (a lone workgroup there hides less: a quarter more),
    and every split's sums go through memory, the more the more rows there are.  Large matrices, which come in pairs, have
    two.  us for 1, 32 and 64 rows by splits: 17408 x 5120 twice 1: 50 73 86, 2: 52 62 75, 4: 49 67 85; 5120 x 17408 6: 34 44 49, 8: 32 41 48,
    12: 34 39 46; 6144, 1024 and 1024 x 5120 4: 16 23 30, 5: 16 23 31, 7: 16 26 32; 1024 x 5120 5: 10 13 22, 10: 8 12 18."""
    v, blocks = visits(cols), -(-rows // 16)
    fits = [s for s in range(1, 17) if -(-v // s) * (s - 1) < v and -(-v // s) <= 63]
    if blocks >= 768:
        return next((s for s in fits if s >= (2 if blocks < 4096 else 1)), fits[-1])

    def cost(s):
        groups = -(-blocks // 8) * s
        return -(-groups // 256) * -(-v // s) * (1.25 if groups <= 256 else 1) + s * (0.2 + blocks / 2560)

    return min(fits, key=cost)


class Planes:
    """The device arrays of one matrix and the structure the kernels take."""

    ARRAYS = ("planes", "bases", "listed_at", "listed")

    def __init__(self, rows, cols, arrays):
        self.rows, self.cols, self.arrays = rows, cols, arrays
        self.splits = sum_splits(rows, cols)
        self.struct = _hip_abi.GrfPlanes(*(arrays[name].data_ptr() for name in self.ARRAYS), rows, cols, self.splits)
        self.address = ctypes.addressof(self.struct)
        self.nbytes = sum(a.numel() * a.element_size() for a in arrays.values())
        self._workspace = {}

    @classmethod
    def of_words(cls, words, launch):
        """Of a dense matrix of BF16 words on the device.  ``launch(function, *arguments)`` adds the stream."""
        import torch
        lib = _native.hip()
        rows, cols = words.shape
        make = lambda n, kind: torch.empty(n, device=words.device, dtype=kind)
        count = lib.grf_planes_visits(rows, cols)
        bases, counts = make(-(-rows // 16) * 16, torch.int32), make(count, torch.int32)
        launch(lib.grf_planes_count, words.data_ptr(), rows, cols, bases.data_ptr(), counts.data_ptr())
        listed_at = torch.zeros(count + 1, device=words.device, dtype=torch.int32)
        torch.cumsum(counts, 0, out=listed_at[1:])
        listed = torch.zeros(int(listed_at[-1]) + 1, device=words.device, dtype=torch.int32)  # (the last is nobody's)
        planes = make(lib.grf_planes_bytes(rows, cols), torch.uint8)
        launch(lib.grf_planes_fill, words.data_ptr(), rows, cols, bases.data_ptr(), listed_at.data_ptr(), planes.data_ptr(), listed.data_ptr())
        return cls(rows, cols, {"planes": planes, "bases": bases, "listed_at": listed_at, "listed": listed})

    def clone(self):
        return Planes(self.rows, self.cols, {k: v.clone() for k, v in self.arrays.items()})

    def workspace(self, m):
        """Bytes a product of ``m`` rows needs."""
        m = min(m, 128)
        if m not in self._workspace:
            self._workspace[m] = int(_native.hip().grf_planes_workspace_bytes(1, ctypes.byref(ctypes.pointer(self.struct)), m))
        return self._workspace[m]
