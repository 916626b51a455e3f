"""The work that users of this library have it do, as cases that can be timed.

What a case stands for is its ``path``:

* ``linear``  ``BctxLinear.forward`` on one coded matrix.  One row is a decode step, 2..8 rows a
              speculative verify pass (``invariant``: rows bit-equal whatever the batch), up to 128
              a batch server's step, more a prompt (prefill).
* ``group``   sibling projections that take the same rows (q/k/v, gate/up) in one launch.
* ``ppcx``    the product of a predictive (PPCX) weight that keeps its reference's contexts.
* ``embed``   ``BctxEmbedding.forward``: rows of a coded table by index.
* ``dense``   ``decode()`` of a coded matrix on the device.
* ``encode``  ``bitexact_context_codec.encode`` on the host: building a package.
* ``restore`` ``bitexact_context_codec.decode`` on the host: verifying and restoring one.
* ``load``    frame bytes on the host -> a tensor resident on the device (what loading a model does
              for every matrix), the dense words read back from it as the result.

Weights look like a model's: N(0, 0.02) times a log-normal scale per row, a thousandth of them
ten times larger.  Products and lookups keep one set of weights per shape, as a loaded model
does, and every state holds device buffers of its own, so that consecutive passes do not find
them in the caches (a model's layers do not either); what the seed draws there are the
activations and the row ids.  Where the coded matrix itself is the input (``dense``, ``encode``,
``restore``, ``load``), the seed draws the matrix.
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from georefine_amd import bitexact_context_codec as codec
from georefine_amd import bitexact_predictive_codec as predictive
from georefine_amd.bitexact_context_gpu import HipContextTensor, HipLinearGroup
from georefine_amd.bitexact_predictive_gpu import HipPredictiveTensor
from georefine_amd.serving import BctxEmbedding, BctxLinear

LARGEST = 5120 * 17408  # weights of the largest matrix of the configurations


def listed():
    return [
        # the smallest product: one token through a k or v projection
        {"name": "one_row_small", "path": "linear", "rows": 1024, "cols": 5120, "m": 1, "invariant": False, "bias": False,
         "block": 0},
        # one token through gate and up, the largest launch of a decode step
        {"name": "one_row_gate_up", "path": "group", "rows": 17408, "rows2": 17408, "rows3": 0, "cols": 5120, "m": 1,
         "invariant": False, "block": 0},
        # verify pass of five draft tokens + 1 through the down projection, rows bit-equal to single-row decoding
        {"name": "verify_down", "path": "linear", "rows": 5120, "cols": 17408, "m": 6, "invariant": True, "bias": False,
         "block": 0},
        # a batch server with 32 users: q, k and v
        {"name": "batch_qkv", "path": "group", "rows": 6144, "rows2": 1024, "rows3": 1024, "cols": 5120, "m": 32,
         "invariant": False, "block": 16},
        # and with 64 users: gate and up
        {"name": "batch_gate_up", "path": "group", "rows": 17408, "rows2": 17408, "rows3": 0, "cols": 5120, "m": 64,
         "invariant": False, "block": 16},
        # prefill of a prompt of 1000 tokens
        {"name": "prompt_down", "path": "linear", "rows": 5120, "cols": 17408, "m": 1000, "invariant": False, "bias": True,
         "block": 0},
        # a whole matrix decoded to dense BF16 (o projection)
        {"name": "dense_o", "path": "dense", "rows": 5120, "cols": 6144},
        # a prompt's rows of an embedding table
        {"name": "embed_prompt", "path": "embed", "rows": 8192, "cols": 5120, "m": 777},
        # 16 users x (5 draft tokens + 1) through a predictive weight
        {"name": "predictive_96", "path": "ppcx", "rows": 4096, "cols": 4096, "m": 96},
        # packaging, restoring and loading, on host data
        {"name": "encode_host", "path": "encode", "rows": 2048, "cols": 5120},
        {"name": "restore_host", "path": "restore", "rows": 1500, "cols": 4304},
        {"name": "load_square", "path": "load", "rows": 4096, "cols": 4096},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _shape(rng, most, step, rows_from=256, cols_from=512):
    """rows (any number, odd ones too) and cols (a multiple of ``step``) with at most ``most`` weights."""
    cols = _log_int(rng, cols_from, 17408) // step * step
    return _log_int(rng, rows_from, min(17408, most // cols)), cols


def draw(rng):
    path = rng.choice(("linear", "linear", "linear", "group", "group", "ppcx", "embed", "dense", "encode", "restore", "load"))
    # widths are mostly multiples of 64; every multiple of 16 (PPCX: 32) is served by the fused kernels
    step = 64 if rng.random() < 0.75 else 16
    if path == "linear":
        rows, cols = _shape(rng, LARGEST // 2, step)
        m = 1 if rng.random() < 0.25 else _log_int(rng, 1, 1000)
        return {"path": path, "rows": rows, "cols": cols, "m": m, "invariant": m <= 128 and rng.random() < 0.3,
                "bias": rng.random() < 0.3, "block": 16 if m >= 16 else 0}
    if path == "group":
        rows, cols = _shape(rng, LARGEST // 4, 64)
        rows2 = rows if rng.random() < 0.5 else _log_int(rng, 256, rows)
        m = 1 if rng.random() < 0.4 else _log_int(rng, 1, 128)
        return {"path": path, "rows": rows, "rows2": rows2, "rows3": rows2 if rng.random() < 0.4 else 0, "cols": cols, "m": m,
                "invariant": rng.random() < 0.3, "block": 16 if m >= 16 else 0}
    if path == "ppcx":
        rows, cols = _shape(rng, 4096 * 4096, max(step, 32))
        return {"path": path, "rows": rows, "cols": cols, "m": _log_int(rng, 1, 128)}
    if path == "embed":
        rows, cols = _shape(rng, 8192 * 5120, step, rows_from=1024)
        return {"path": path, "rows": rows, "cols": cols, "m": _log_int(rng, 1, 2048)}
    # where the seed draws the matrix itself
    rows, cols = _shape(rng, 5120 * 6144 if path == "dense" else 2048 * 5120, step)
    return {"path": path, "rows": rows, "cols": cols}


# ------------------------------------------------------------------- inputs

def _generator(*numbers):
    g = torch.Generator(device="cuda")
    seed = 0x9E3779B9
    for n in numbers:
        seed = (seed * 1000003 + int(n) + 1) % (1 << 62)
    g.manual_seed(seed)
    return g


def _weights(g, rows, cols):
    w = torch.randn(rows, cols, device="cuda", generator=g)
    w *= 0.02 * torch.exp(0.5 * torch.randn(rows, 1, device="cuda", generator=g))
    return torch.where(torch.rand(rows, cols, device="cuda", generator=g) < 1e-3, 10.0 * w, w)


def _words(w):
    return w.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16)


def _activations(g, m, cols):
    return torch.randn(m, cols, device="cuda", generator=g).bfloat16()


_resident = {}  # the model: one coded tensor per shape and member


def _context_tensors(shapes, segment=None):
    """The model's coded matrices of these shapes, one per member; frames are built side by side."""
    todo = [(i, r, c) for i, (r, c) in enumerate(shapes) if ("bctx", i, r, c, segment) not in _resident]
    words = [_words(_weights(_generator(17, i, r, c), r, c)) for i, r, c in todo]

    def build(w):
        frame = codec.encode(w, residual="raw6")
        return frame, HipContextTensor.host_prepare(frame, fused_segment=segment)

    with ThreadPoolExecutor(max_workers=4) as pool:
        built = list(pool.map(build, words))
    for (i, r, c), (frame, prepared) in zip(todo, built):
        _resident["bctx", i, r, c, segment] = HipContextTensor(frame, device="cuda:0", fused_segment=segment, prepared=prepared)
    return [_resident["bctx", i, r, c, segment] for i, (r, c) in enumerate(shapes)]


def _predictive_tensor(rows, cols):
    key = ("ppcx", rows, cols)
    if key not in _resident:
        g = _generator(18, rows, cols)
        w = _weights(g, rows, cols)
        target = _words(w)
        reference = _words(w.bfloat16().float() + 0.002 * torch.randn(rows, cols, device="cuda", generator=g))
        _resident[key] = HipPredictiveTensor(predictive.encode(target, reference), reference, device="cuda:0")
    return _resident[key]


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.path = path = case["path"]
    rows, cols = case["rows"], case["cols"]
    g = _generator(19, seed)
    if path == "linear":
        s.module = BctxLinear(_context_tensors([(rows, cols)])[0].clone(residual_block=case["block"] or None),
                              torch.nn.Parameter(_activations(g, 1, rows)[0], requires_grad=False) if case["bias"] else None,
                              batch_invariant=case["invariant"])
        s.x = _activations(g, case["m"], cols)
    elif path == "group":
        shapes = [(r, cols) for r in (rows, case["rows2"], case["rows3"]) if r]
        s.group = HipLinearGroup([t.clone(residual_block=case["block"] or None) for t in _context_tensors(shapes, 64)])
        s.invariant = case["invariant"]
        s.x = _activations(g, case["m"], cols)
    elif path == "ppcx":
        s.tensor = _predictive_tensor(rows, cols).clone()
        s.x = _activations(g, case["m"], cols)
    elif path == "embed":
        s.module = BctxEmbedding(_context_tensors([(rows, cols)])[0].clone())
        s.ids = torch.randint(0, rows, (case["m"],), device="cuda", generator=g)
    elif path == "encode":
        s.words = _words(_weights(g, rows, cols))
    else:
        words = _words(_weights(g, rows, cols))
        s.frame = codec.encode(words, residual="raw6" if path == "dense" else "auto")
        if path == "dense":
            s.tensor = HipContextTensor(s.frame, device="cuda:0")
    return s


def run(s):
    if s.path == "linear":
        return s.module(s.x)
    if s.path == "group":
        return s.group.linear(s.x, batch_invariant=s.invariant)
    if s.path == "ppcx":
        return s.tensor.linear(None, s.x)
    if s.path == "embed":
        return s.module(s.ids).view(torch.int16)
    if s.path == "dense":
        return s.tensor.decode(check=False).view(torch.int16)
    if s.path == "encode":
        frame = codec.encode(s.words)
        out = np.zeros(2 * s.words.size + 256, dtype=np.uint8)  # (one length whatever the seed: frames are never longer)
        out[:len(frame)] = np.frombuffer(frame, dtype=np.uint8)
        return out
    if s.path == "restore":
        return codec.decode(s.frame).view(np.int16)
    return HipContextTensor(s.frame, device="cuda:0").decode().view(torch.int16)


# ------------------------------------------------------------------- what it is measured against

CODED = 10.5 / 8        # bytes per weight of a context frame of such weights
PREDICTIVE = 7.9 / 8    # of a predictive frame ...
CONTEXTS = 4 / 8        # ... and of the contexts it is decoded with


def work(case):
    rows, cols, m = case["rows"], case["cols"], case.get("m", 0)
    n = rows * cols
    if case["path"] == "group":
        total = rows + case["rows2"] + case["rows3"]
        return {"bytes": total * cols * CODED + 2 * m * (cols + total), "flops": 2 * m * total * cols}
    if case["path"] == "linear":
        return {"bytes": n * CODED + 2 * m * (cols + rows), "flops": 2 * m * n}
    if case["path"] == "ppcx":
        return {"bytes": n * (PREDICTIVE + CONTEXTS) + 2 * m * (cols + rows), "flops": 2 * m * n}
    if case["path"] == "embed":
        return {"bytes": m * cols * (CODED + 2) + 8 * m, "flops": 0}
    return {"bytes": n * (CODED + 2), "flops": 0}


def tolerance(case):
    # products: fp32 sums of exact BF16 products, rounded once to BF16; everything else is the weights' own bits
    return {"rel": 5e-3} if case["path"] in ("linear", "group", "ppcx") else "exact"
