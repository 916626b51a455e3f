"""Times forced tilings of the matrix-core products, for the planner's fitted model (``_fused.gemm_times``):

    python profiles/gemm_tilings.py OUT.csv [SEED]

One line per tiling: the matrix, what ``gemm_times`` is given, and us a call among others (three copies of the
matrix in turn) at 2 to 128 rows.  ``chosen``: s for the slot model's choice, p for the tiling that ``gemm_times``
promises most of against it, before ``gain_to_ask`` has its say.  ``part``: "sweep", matrices with many
tilings each, which say how far the model is off; "pair", matrices drawn over the sizes that are served, with these
two alone where they differ, which say where the lines of ``gain_to_ask`` lie.  Every tiling is checked by the
library's host-side validator before it is launched.
"""
import csv
import math
import os
import random
import sys
from pathlib import Path

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
import numpy as np
import torch

from georefine_amd import _fused, _planes, bitexact_context_codec as codec
from georefine_amd.bitexact_context_gpu import HipContextTensor

_planes.FROM_WEIGHTS = 1 << 40  # what is timed is the walk: matrices of every size stay frames

NAMED = [(300, 4096), (450, 6144), (600, 5120), (1024, 5120), (1500, 2064), (700, 9216), (2048, 5120), (2560, 5120), (3000, 3072),
         (4096, 4096), (5120, 6144), (6144, 5120), (5120, 17408), (17408, 5120)]
ROWS = (2, 6, 20, 32, 50, 64, 100, 128)


def matrices():
    """(part, rows, cols, tilings at most beside the two choices)."""
    rng = random.Random(11)
    whole = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    def drawn():
        step = 64 if rng.random() < 0.75 else 16
        cols = max(512, whole(512, 17408) // step * step)
        return whole(128, min(17408, (44 << 20) // cols)), cols

    return ([("sweep", rows, cols, 50) for rows, cols in NAMED] + [("sweep", *drawn(), 30) for _ in range(30)]
            + [("pair", *drawn(), 0) for _ in range(1200)])


def frame_of(rows, cols):
    g = torch.Generator(device="cuda").manual_seed(rows * cols)
    w = torch.randn(rows, cols, device="cuda", generator=g) * 0.02 * torch.exp(0.5 * torch.randn(rows, 1, device="cuda", generator=g))
    w = torch.where(torch.rand(rows, cols, device="cuda", generator=g) < 1e-3, 10.0 * w, w)
    return codec.encode(w.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16), residual="raw6")


def candidates(plan, rng):
    """(lanes per row, rows, parts) of tilings with four waves at least: whole blocks of sixteen rows, or cut once
    more by the workgroup slots they leave."""
    counts, found = _fused._tile_counts(plan.class_rows, 1024), {}
    for quads in range(2, -(-plan.spr // 4) + 1):
        for blocks in range(1, 17):
            p, r = min(4 * quads, plan.spr), 16 * blocks
            threads = _fused.gemm_shape(p, r)[2]
            if not 256 <= threads <= 1024:
                continue
            for k in _fused.GEMM_K_PARTS:
                if k <= -(-plan.spr // p):
                    for slots in (256, 512, 768):
                        found[p, _fused._spread_rows(counts, r, max(slots // k, counts[r]), 16 * (blocks - 1) + 1), k] = True
                    found[p, r, k] = True
    found = list(found)
    rng.shuffle(found)
    return found


GIVEN = ("threads", "tallest", "blocks", "n_slabs", "tiles", "k", "lds")


def forced(plan, choice):
    os.environ["GEOREFINE_FUSED_GEMM_TILING"] = ",".join(map(str, choice))
    try:
        return plan.gemm_tiling()
    finally:
        del os.environ["GEOREFINE_FUSED_GEMM_TILING"]


def columns(plan, t):
    """What ``gemm_times`` is given for a tiling."""
    g = t["scalars"]
    k = max(1, g["k_parts"])
    tall = -(-g["rows_per_tile"] // 16)
    blocks = _fused._blocks_paid(t["tile_rows"], g["rows_per_tile"]) * k / g["n_tiles"] if tall > 1 else 1.0
    return dict(threads=g["threads"], lanes=g["lanes_per_row"], rows_per_tile=g["rows_per_tile"], tallest=tall, blocks=round(blocks, 4),
                n_slabs=g["n_slabs"], tiles=g["n_tiles"], k=k, lds=t["lds"])


def time_us(copies, x):
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = float("inf")
    for _ in range(7):
        for i in range(3):
            copies[i % len(copies)].gemm(x)
        begin.record()
        for i in range(24):
            copies[i % len(copies)].gemm(x)
        end.record()
        end.synchronize()
        best = min(best, begin.elapsed_time(end) * 1000 / 24)
    return best


def modelled(plan, t):
    given = columns(plan, t)
    return float(np.log(_fused.gemm_times(*(np.array([given[key]]) for key in GIVEN), plan.spr, plan.seg_len, plan.table_bytes())).mean())


def most_promised(plan):
    asked = _fused.gain_to_ask
    _fused.gain_to_ask = lambda threads, tiles, k, lds, rows, cus=256: np.full(len(k), 0.05)
    try:
        return plan._gemm_tiling(True)
    finally:
        _fused.gain_to_ask = asked


def tilings(plan, rng, most):
    """[(chosen, tiling)]: the two choices, then the best by the model, then others at random."""
    slot, promised = plan.gemm_tiling(False), most_promised(plan)
    todo, made = [("s", slot)] + ([] if slot["scalars"] == promised["scalars"] else [("p", promised)]), []
    seen = [t["scalars"] for _, t in todo]
    for choice in candidates(plan, rng) if most else ():
        if len(made) >= 3 * most:
            break
        try:
            t = forced(plan, choice)
        except _fused.FusedUnsupported:
            continue  # does not fit in LDS
        if t["scalars"] not in seen:
            seen.append(t["scalars"])
            made.append(("", t))
    best = sorted(range(len(made)), key=lambda i: modelled(plan, made[i][1]))[:most // 2]
    return todo + [made[i] for i in best] + [t for i, t in enumerate(made) if i not in best][:most - most // 2]


def main():
    out, rng = sys.argv[1], random.Random(int(sys.argv[2]) if len(sys.argv) > 2 else 1)
    writer = None
    with open(out, "w", newline="") as file:
        for part, rows, cols, most in matrices():
            tensor = HipContextTensor(frame_of(rows, cols), device="cuda:0")
            plan = tensor._plan
            block, position, _ = plan.residual_order()
            todo = tilings(plan, rng, most)
            if part == "pair" and len(todo) < 2:
                continue
            copies = [tensor] + [tensor.clone() for _ in range(2)]
            xs = [torch.randn(m, cols, device="cuda").bfloat16() for m in ROWS]
            for _ in range(100):  # (the clock has to come up)
                tensor.gemm(xs[-1])
            for chosen, t in todo:
                _fused.validate_host(plan, t, "gemm", row_pos=position, block=block)
                tensor._tilings.pop("gemm", None)
                plan.gemm_tiling = lambda t=t: t
                try:
                    uploaded = tensor._gemm_tiling()
                finally:
                    del plan.gemm_tiling
                for c in copies:
                    c._tilings["gemm"] = uploaded
                line = dict(part=part, rows=rows, cols=cols, spr=plan.spr, seg_len=plan.seg_len, table_bytes=plan.table_bytes(),
                            chosen=chosen, **columns(plan, t), **{f"us_{m}": round(time_us(copies, x), 2) for m, x in zip(ROWS, xs)})
                if writer is None:
                    writer = csv.DictWriter(file, line)
                    writer.writeheader()
                writer.writerow(line)
                file.flush()
            print(part, rows, cols, "seg", plan.seg_len, "tilings", len(todo), flush=True)


if __name__ == "__main__":
    main()
