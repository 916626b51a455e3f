"""Times both sides of two of the planner's choices over matrices drawn from the sizes that are served:

    python profiles/planner_choices.py lookups OUT.csv [SEED]
    python profiles/planner_choices.py lines OUT.csv [SEED]

``lookups``: products of a predictive weight on the matrix cores with 64 KiB of lookups and with 16 KiB
(``FramePlan.for_matrix_cores``), us a call among others at 2 to 128 rows.  ``lines``: decode to dense with the GEMV's
tiling and with that of the kernel that stores whole lines (``FramePlan.lines_tiling``), by how many results are written
in turn (one stays in the last-level cache while it fits, four do not).  One line per matrix, with the
tilings and what the planner's model says of them.  predictive_lookups.csv holds such a run and one over
more matrices where three workgroups share a unit.
"""
import collections
import csv
import math
import random
import sys
from pathlib import Path

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
import numpy as np
import torch

from georefine_amd import _fused, _planes, bitexact_context_codec as codec, bitexact_predictive_codec as predictive
from georefine_amd.bitexact_context_gpu import HipContextTensor
from georefine_amd.bitexact_predictive_gpu import HipPredictiveTensor

_planes.FROM_WEIGHTS = 1 << 40  # what is timed is the walk: matrices of every size stay frames

ROWS = (2, 6, 20, 32, 64, 96, 128)


def weights(rows, cols):
    g = torch.Generator(device="cuda").manual_seed(rows * cols)
    w = torch.randn(rows, cols, device="cuda", generator=g) * 0.02 * torch.exp(0.5 * torch.randn(rows, 1, device="cuda", generator=g))
    return torch.where(torch.rand(rows, cols, device="cuda", generator=g) < 1e-3, 10.0 * w, w), g


def words(w):
    return w.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16)


def both_us(sides, launches=20):
    """us a call of each side, the sides in turn, three copies of the matrix in turn: the best of seven."""
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = [float("inf")] * len(sides)
    for _ in range(7):
        for i, call in enumerate(sides):
            for j in range(3):
                call(j)
            begin.record()
            for j in range(launches):
                call(j % 3)
            end.record()
            end.synchronize()
            best[i] = min(best[i], begin.elapsed_time(end) * 1000 / launches)
    return [round(v, 2) for v in best]


def described(name, tiling):
    return {f"{name}_{key}": tiling["scalars"].get(key, 0) if key != "lds" else tiling["lds"]
            for key in ("threads", "lanes_per_row", "rows_per_tile", "n_slabs", "n_tiles", "k_parts", "lds")}


def predictive_matrices(rng):
    whole = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    yield from [(4096, 4096), (8192, 2048), (16384, 1024), (3152, 4544), (1624, 4800), (1092, 12480), (2048, 8192)]
    for _ in range(60):  # about where three workgroups share a unit
        cols = 64 * rng.choice((rng.randint(12, 16), rng.randint(24, 32), rng.randint(52, 64)))
        yield whole((13 << 20) // cols, min(17408, (17 << 20) // cols)), cols
    for _ in range(240):
        step = 64 if rng.random() < 0.75 else 32
        cols = max(512, whole(512, 17408) // step * step)
        rows = whole(512, min(17408, (16 << 20) // cols))
        if rows * cols >= 3 << 20:
            yield rows, cols


def lookups(rng):
    choice = _fused.FramePlan.for_matrix_cores
    for rows, cols in predictive_matrices(rng):
        w, g = weights(rows, cols)
        reference = words(w.bfloat16().float() + 0.002 * torch.randn(rows, cols, device="cuda", generator=g))
        frame, sides = predictive.encode(words(w), reference), []
        _fused.FramePlan.for_matrix_cores = lambda plan, *a: plan
        try:
            sides.append(HipPredictiveTensor(frame, reference, device="cuda:0"))
            plan = sides[0]._plan
            if plan is None:
                continue
            _fused.FramePlan.for_matrix_cores = _fused.FramePlan.with_lookups
            sides.append(HipPredictiveTensor(frame, reference, device="cuda:0"))
        finally:
            _fused.FramePlan.for_matrix_cores = choice
        other = sides[1]._matrix_plan
        tall, fitted, fine = plan.gemm_tiling(False), plan.gemm_tiling(True), other.gemm_tiling(False)
        g = fine["scalars"]
        if g["n_tiles"] <= 256 or _fused.lds_share(fine["lds"]) < 2:  # (a workgroup a unit on either side)
            continue
        copies = [[t, t.clone(), t.clone()] for t in sides]
        line = dict(rows=rows, cols=cols, seg_len=plan.seg_len, share_64=round(plan.gemm_share(tall), 4),
                    share_64_fitted=round(plan.gemm_share(fitted), 4), share_16=round(other.gemm_share(fine), 4),
                    **described("slot", tall), **described("fitted", fitted), **described("small", fine))
        for m in ROWS:
            x = torch.randn(m, cols, device="cuda").bfloat16()
            line[f"us64_{m}"], line[f"us16_{m}"] = both_us([lambda j, c=c: c[j].linear(None, x) for c in copies])
        yield line


def whole_lines(rng):
    whole = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    named = [(5120, 6144), (17408, 5120), (5120, 17408), (2560, 5120), (9000, 2048), (8192, 5120), (4096, 4096), (11580, 2048)]
    rule = _fused.wave_time
    for n in range(360):
        cols = max(512, whole(512, 17408) // 64 * 64)
        rows, cols = named[n] if n < len(named) else (whole(256, min(17408, (44 << 20) // cols)), cols)
        tensor = HipContextTensor(codec.encode(words(weights(rows, cols)[0]), residual="raw6"), device="cuda:0")
        plan = tensor._plan
        if plan is None or plan.seg_len % 64:
            continue
        plan._tilings.pop(("lines", None), None)
        _fused.wave_time = lambda *a, **k: 1.0
        try:
            lines = plan.lines_tiling()
        finally:
            _fused.wave_time = rule
        walk = plan.tiling(1, waves=True)
        copies = [[tensor.clone() for _ in range(3)] for _ in range(2)]
        for c in copies[0]:
            c._store_tiling = lambda c=c: c._tiling(1)
        for c in copies[1]:
            c._tilings.pop("lines", None)
            c._upload_tiling("lines", lines)
        us = {}
        for results in (1, 2, 4):  # how many the program writes in turn: a result's buffer is free once no one holds it
            kept = collections.deque(maxlen=results - 1)
            us[results] = both_us([lambda j, c=c: kept.append(c[j].decode(check=False)) for c in copies])
        yield dict(rows=rows, cols=cols, seg_len=plan.seg_len, model_walk=round(rule(walk, plan.seg_len, plan.table_bytes()), 1),
                   model_lines=round(rule(lines, plan.seg_len, plan.table_bytes(), waves=_fused.LINES_WAVES_PER_CU), 1),
                   **described("walk", walk), **described("lines", lines),
                   **{f"us_{name}_{n}": us[n][i] for n in us for i, name in enumerate(("walk", "lines"))})


def main():
    rng, writer = random.Random(int(sys.argv[3]) if len(sys.argv) > 3 else 1), None
    with open(sys.argv[2], "w", newline="") as file:
        for line in {"lookups": lookups, "lines": whole_lines}[sys.argv[1]](rng):
            if writer is None:
                writer = csv.DictWriter(file, line)
                writer.writeheader()
            writer.writerow(line)
            file.flush()
            print(line["rows"], line["cols"], flush=True)


if __name__ == "__main__":
    main()
