"""Prompts and embedding lookups for a profiler (summarize.py):

    python3 profiles/prompts.py {prompt,lookup} [--steps N] [--warmup N] [--calibrate-copy] [--walked]

``prompt``: 1000 activation rows of a coded 5120 x 17408 matrix (``--walked``: decode to dense, then the product).  ``lookup``: 777 rows of a
coded 8192 x 5120 table.  Three device copies of the matrix in turn, eager calls.  Prints one line of JSON.
"""
import argparse
import json
import sys
from pathlib import Path

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
import numpy as np
import torch

import bench
from georefine_amd import _planes, bitexact_context_codec as codec
from georefine_amd.bitexact_context_gpu import HipContextTensor

SIZES = {"prompt": (5120, 17408, 1000), "lookup": (8192, 5120, 777)}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("what", choices=SIZES)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--calibrate-copy", action="store_true")
    ap.add_argument("--walked", action="store_true", help="the matrix stays a frame")
    args = ap.parse_args()
    if args.walked:
        _planes.FROM_WEIGHTS = 1 << 40
    rows, cols, m = SIZES[args.what]
    g = torch.Generator(device="cuda").manual_seed(1)
    w = torch.randn(rows, cols, device="cuda", generator=g) * 0.02 * torch.exp(0.5 * torch.randn(rows, 1, device="cuda", generator=g))
    w = torch.where(torch.rand(rows, cols, device="cuda", generator=g) < 1e-3, 10.0 * w, w)
    t = HipContextTensor(codec.encode(w.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16), residual="raw6"))
    copies = [t, t.clone(), t.clone()]
    if args.what == "prompt":
        xs = [torch.randn(m, cols, device="cuda", generator=g).bfloat16() for _ in copies]
        call = lambda i: copies[i % 3].linear(xs[i % 3])
    else:
        ids = [torch.randint(0, rows, (m,), device="cuda", generator=g) for _ in copies]
        call = lambda i: copies[i % 3].gather_rows(ids[i % 3])
    for i in range(args.warmup):
        call(i)
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    begin.record()
    for i in range(args.steps):
        call(i)
    end.record()
    end.synchronize()
    if args.calibrate_copy:
        bench.calibration_copy(torch)
        torch.cuda.synchronize()
    print(json.dumps({"metric": f"{args.what}, us a call", "value": round(begin.elapsed_time(end) * 1000 / args.steps, 2)}))


if __name__ == "__main__":
    main()
