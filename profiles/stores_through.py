"""Decode to dense with the results stored through to what the device shares, and kept by the second-level caches:

    python profiles/stores_through.py build FOLDER
    python profiles/stores_through.py measure FOLDER OUT.csv [SEED]
    python profiles/stores_through.py predictive FOLDER OUT.csv [SEED]
    python profiles/stores_through.py lookups FOLDER OUT.csv [SEED]

FOLDER/through.so and FOLDER/kept.so are the library with the one and with the other whatever the size
(the rules of ``launch_wave_store`` and ``launch_gather`` taken out).  us a decode as replays of one graph, four coded matrices and four results in turn, alone and
with a product of 256 rows after each decode, the sides in turn; matrices are drawn over the sizes that are served.
stores_through.csv holds runs with seeds 1 to 4, of which 3 and 4 draw columns that end between lines.
``predictive``: the same of predictive weights, results of 6 MiB and more; predictive_stores_through.csv holds a run with seed 1.
``lookups``: the same of a row gather, us a launch in a graph, alone and with a sum over its rows after it, and us a whole call that tells of
errors: rows kept and a wait for the stream, or rows past the caches and the word polled.  lookups_through.csv holds runs with seeds 1, 2 and 3, of which the
last is of 400 to 1300 rows, about as many as there are places for on the compute units.
"""
import csv
import ctypes
import math
import random
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))
LINES = {"const bool far = (uint64_t)f.rows * f.cols * 2 < below << 20 && !": "const bool far = (void(below), {}) && !",
         "const bool far = f.seg_len % 32 == 0 && (uint64_t)count * f.cols * 2 < 64u << 20;": "const bool far = {};"}
SIDES = {"kept": "false", "through": "true"}
NAMED = [(1024, 1024), (2048, 2048), (4096, 2048), (4096, 4096), (1024, 5120), (2048, 5120), (5120, 4096), (5120, 6144)]


def build(folder):
    from georefine_amd import _native
    for side, rule in SIDES.items():
        with tempfile.TemporaryDirectory() as scratch:
            for path in (ROOT / "georefine_amd/csrc").glob("*.h*"):
                text = path.read_text()
                if path.name == "fused_kernels.h":
                    for line, instead in LINES.items():
                        assert text.count(line) == 1
                        text = text.replace(line, instead.format(rule))
                (Path(scratch) / path.name).write_text(text)
            flags = ["hipcc", *_native.HIP_FLAGS, "-I", str(ROOT / "include")]
            objects = [str(Path(scratch) / (path.stem + ".o")) for path in _native.hip_sources()]
            with ThreadPoolExecutor() as pool:
                list(pool.map(lambda to: subprocess.run([*flags, "-c", to[:-2] + ".hip", "-o", to], check=True), objects))
            subprocess.run(["hipcc", "-shared", f"--offload-arch={_native.HIP_ARCH}", *objects, "-o", str(Path(folder) / (side + ".so"))],
                           check=True)


def drawn(rng, ragged):
    """Up to 96 MiB of result, most of them below 48; ragged: columns that allow segments of 16 or 32 only, 2 MiB and more."""
    whole = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if ragged:
        cols = whole(256, 17408) // 64 * 64 + rng.choice((16, 32, 32))
        return min(17408, whole(2 << 20, 64 << 20) // (2 * cols)), cols
    cols = max(256, whole(256, 17408) // 64 * 64 if rng.random() < 0.75 else whole(256, 17408) // 16 * 16)
    return whole(64, max(65, min(17408, (48 << 20) // cols))), cols


def drawn_predictive(rng):
    whole = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    cols = whole(512, 17408) // 64 * 64 + rng.choice((0, 32))
    return min(17408, whole(6 << 20, 60 << 20) // (2 * cols)), cols


def libraries(folder):
    from georefine_amd import _hip_abi
    libs = {side: ctypes.CDLL(str((Path(folder) / (side + ".so")).resolve())) for side in SIDES}
    for lib in libs.values():
        _hip_abi.declare(lib)
    return libs


def coded(rows, cols):
    import numpy as np
    import torch
    from georefine_amd import _planes, bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor
    _planes.FROM_WEIGHTS = 1 << 40  # what is timed is the walk: matrices of every size stay frames
    g = torch.Generator(device="cuda").manual_seed(rows * cols)
    w = torch.randn(rows, cols, device="cuda", generator=g) * 0.02 * torch.exp(0.5 * torch.randn(rows, 1, device="cuda", generator=g))
    w = torch.where(torch.rand(rows, cols, device="cuda", generator=g) < 1e-3, 10.0 * w, w)
    return HipContextTensor(codec.encode(w.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16), residual="raw6"))


def coded_predictive(rows, cols):
    import numpy as np
    import torch
    from georefine_amd import _planes, bitexact_predictive_codec as predictive
    from georefine_amd.bitexact_predictive_gpu import HipPredictiveTensor
    _planes.FROM_WEIGHTS = 1 << 40  # (as in coded)
    g = torch.Generator(device="cuda").manual_seed(rows * cols)
    w = torch.randn(rows, cols, device="cuda", generator=g) * 0.02 * torch.exp(0.5 * torch.randn(rows, 1, device="cuda", generator=g))
    near = w + 0.002 * torch.randn(rows, cols, device="cuda", generator=g)
    w, near = (v.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16) for v in (w, near))
    return HipPredictiveTensor(predictive.encode(w, near), near, device="cuda:0")


def best_us(graphs, launches, rounds=9):
    """us a launch of each graph, the graphs in turn."""
    import torch
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = [math.inf] * len(graphs)
    for _ in range(rounds):
        for k, graph in enumerate(graphs):
            graph.replay()
            begin.record()
            graph.replay()
            graph.replay()
            end.record()
            end.synchronize()
            best[k] = min(best[k], begin.elapsed_time(end) * 1000 / (2 * launches))
    return best


def lookups(folder, out, seed):
    import time
    import torch
    from georefine_amd import bitexact_context_gpu as gpu
    libs = libraries(folder)
    rng, launches = random.Random(seed), 12
    whole = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    tables = [(8192, 5120), (32768, 1024)] if seed == 1 else []
    while len(tables) < 40:
        cols = whole(512, 17408) // 64 * 64 + rng.choice((0, 0, 16, 32))
        tables.append((whole(1024, min(32768, 8192 * 5120 // cols)), cols))
    with open(out, "w", newline="") as file:
        write = csv.writer(file, lineterminator="\n")
        write.writerow(("rows", "cols", "seg_len", "ids", "lanes", "us_kept", "us_through", "sum_kept", "sum_through", "call_waits", "call_polls"))
        for count, (rows, cols) in enumerate(tables):
            print(count, rows, cols, flush=True)
            t = coded(rows, cols)
            copies = [t, t.clone(), t.clone()]
            spread = {1, whole(2, 200), whole(200, 1000), whole(1000, 3000), whole(3000, 9000)}
            for n in sorted(spread if seed < 3 else {whole(400, 1300) for _ in range(6)}):
                if n * cols > 64 << 20:
                    continue
                ids = [torch.randint(0, rows, (n,), device="cuda") for _ in copies]
                want, graphs = t.gather_rows(ids[0]), []
                for sums in (False, True):
                    for lib in libs.values():
                        def look_up(i):
                            copies[i]._lib = lib
                            return copies[i].gather_rows(ids[i], check=False, validate=False)
                        if not torch.equal(look_up(0), want):
                            sys.exit(f"wrong: {rows} x {cols}, {n}")
                        graph = torch.cuda.CUDAGraph()
                        with torch.cuda.graph(graph):
                            kept = [look_up(i % 3) for i in range(3)]
                            for i in range(launches):
                                copies[i % 3]._lib = lib
                                got = look_up(i % 3)
                                if sums:
                                    got.square_()
                        graphs.append(graph)
                best = best_us(graphs, launches + 3)
                calls = [math.inf] * 2
                for c in copies:
                    c._lib = libs["kept"]
                rule = gpu.gather_polled
                for _ in range(9):
                    for k, polled in enumerate((False, True)):
                        gpu.gather_polled = lambda count, waves, polled=polled: polled
                        for i in range(3):
                            copies[i].gather_rows(ids[i])
                        begin = time.perf_counter()
                        for i in range(18):
                            copies[i % 3].gather_rows(ids[i % 3])
                        calls[k] = min(calls[k], (time.perf_counter() - begin) * 1e6 / 18)
                gpu.gather_polled = rule
                write.writerow((rows, cols, t.fused.seg_len, n, t._gather[0], *(round(v, 2) for v in best + calls)))
            file.flush()


def measure(folder, out, seed, predictive):
    import torch
    from georefine_amd import _native
    from georefine_amd.bitexact_context_gpu import dense_linear
    libs = libraries(folder)
    rng, launches = random.Random(seed), 12
    matrices = (NAMED if seed == 1 else []) + [drawn_predictive(rng) if predictive else drawn(rng, seed > 2)
                                               for _ in range(36 if predictive else 60)]
    with open(out, "w", newline="") as file:
        write = csv.writer(file, lineterminator="\n")
        write.writerow(("rows", "cols", "seg_len", "us_kept", "us_through", "product_kept", "product_through"))
        for count, (rows, cols) in enumerate(matrices):
            print(count, rows, cols, flush=True)
            t = coded_predictive(rows, cols) if predictive else coded(rows, cols)
            if t.fused is None:
                continue
            copies = [t, t.clone(), t.clone(), t.clone()]
            outs = [torch.empty(rows, cols, device="cuda", dtype=torch.bfloat16) for _ in copies]
            x = torch.randn(256, cols, device="cuda").bfloat16()
            want = t.decode(None) if predictive else t.decode()

            def decode(lib, i):
                to = outs[i].data_ptr(), copies[i].error.data_ptr(), torch.cuda.current_stream().cuda_stream
                frame = ctypes.byref(copies[i].fused)
                if predictive:
                    status = lib.grf_ppcx_fused_decode(frame, ctypes.byref(copies[i]._tiling_for("waves")[0]),
                                                       copies[i]._contexts(None)[0].data_ptr(), *to)
                else:
                    status = lib.grf_bctx_fused_decode(frame, ctypes.byref(copies[i]._store_tiling()[0]), *to)
                if status:
                    sys.exit(f"launch: {status}")

            graphs = []
            for product in (False, True):
                for lib in libs.values():
                    decode(lib, 0)
                    dense_linear(_native.hip(), x, outs[0], None, 0)
                    torch.cuda.synchronize()
                    if not torch.equal(outs[0], want):
                        sys.exit(f"wrong: {rows} x {cols}")
                    outs[0].zero_()
                    graph = torch.cuda.CUDAGraph()
                    with torch.cuda.graph(graph):
                        for i in range(launches):
                            decode(lib, i % 4)
                            if product:
                                dense_linear(_native.hip(), x, outs[i % 4], None, 0)
                    graphs.append(graph)
            write.writerow((rows, cols, t.fused.seg_len, *(round(v, 2) for v in best_us(graphs, launches))))
            file.flush()


if __name__ == "__main__":
    if sys.argv[1:2] == ["build"]:
        build(sys.argv[2])
    elif sys.argv[1:2] in (["measure"], ["predictive"]):
        measure(sys.argv[2], sys.argv[3], int(sys.argv[4]) if len(sys.argv) > 4 else 1, sys.argv[1] == "predictive")
    elif sys.argv[1:2] == ["lookups"]:
        lookups(sys.argv[2], sys.argv[3], int(sys.argv[4]) if len(sys.argv) > 4 else 1)
    else:
        sys.exit(__doc__)
