"""The plan of the product over a decoded matrix (``grf_dense_gemm_plan``): its model in Python, and what it is held to.

    python profiles/dense_plan.py build PROBE.so
    python profiles/dense_plan.py tilings PROBE.so OUT.csv [SEED]
    python profiles/dense_plan.py linear OUT.csv [SEED]

``tilings``: every tile, whole and cut along K as the plan considers it, us a product among others (three of W and of x
in turn) as replays of one graph.  PROBE.so is csrc/dense_gemm.hip with an entry point that launches the tile it is asked for.
``linear``: a call of more than 128 rows, decode and product, with the framework's product and with the library's, us a call
among others by eager launches, three copies of the coded matrix and of x in turn, the sides in turn; then the products
alone in the same way.  Matrices and row counts are drawn over the sizes that are served.  dense_tilings.csv holds a run with
seed 1, dense_linear.csv runs with 1, 2 and 3.
"""
import csv
import ctypes
import math
import random
import re
import subprocess
import sys
import tempfile
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))
SOURCE = ROOT / "georefine_amd/csrc/dense_gemm.hip"
NAMED = [(1024, 5120), (5120, 6144), (6144, 5120), (5120, 17408), (17408, 5120), (4096, 4096), (2048, 12288), (6144, 8192)]


# ---------------------------------------------------------------- the model

def constants(text):
    """Tiles (m, n, resident, start, part, full, round, second, sums), units and the least time of a cut product."""
    table = re.search(r"kTiles\[\] = \{(.*?)\};", text, re.S)[1]
    tiles = [tuple(float(v) for v in row.split(",")) for row in re.findall(r"\{([^{}]*)\}", table)]
    return tiles, int(re.search(r"kUnits = (\d+)", text)[1]), float(re.search(r"kCutAtLeast = ([\d.]+)", text)[1])


TILES, UNITS, CUT_AT_LEAST = constants(SOURCE.read_text())


def modelled(tile, parts, rows, cols, m):
    """(parts there are, us) of a product in that tile, cut into at most ``parts``."""
    tile_m, tile_n, resident, start, part, full, each_round, second, sums = TILES[tile]
    steps, tiles = -(-cols // 64), -(-m // int(tile_m)) * -(-rows // int(tile_n))
    per = -(-steps // min(parts, max(1, steps // 2), 64))
    parts = -(-steps // per)
    on_unit = -(-tiles * parts // UNITS)
    us = (start + per * (full * (on_unit // int(resident)) + (part if on_unit % resident else 0.0))
          + each_round * -(-on_unit // int(resident)))
    return parts, max(us + second + sums * 8e-6 * parts * m * rows, CUT_AT_LEAST) if parts > 1 else us


def considered(rows, cols, m):
    """{(tile, parts): us} of what the plan chooses from."""
    found = {}
    for tile, (tile_m, tile_n, resident, *_) in enumerate(TILES):
        tiles = -(-m // int(tile_m)) * -(-rows // int(tile_n))
        for fill in range(int(resident) + 1):
            parts, us = modelled(tile, max(1, UNITS * fill // tiles) if fill else 1, rows, cols, m)
            found.setdefault((tile, parts), us)
    return found


def chosen(rows, cols, m):
    found = considered(rows, cols, m)
    return min(found, key=found.get)


# ---------------------------------------------------------------- measurement

PROBE = """
#include "dense_gemm.hip"
extern "C" int probe_dense(uint32_t tile, uint32_t parts, const uint16_t *w, uint32_t rows, uint32_t cols, const uint16_t *x,
                           uint32_t m_rows, uint16_t *y, void *space, size_t bytes, void *stream) {
  if (tile >= kTileCount || !parts || !dense_fits(rows, cols, m_rows)) return 1;
  const DensePlan p = plan_tile(tile, parts, rows, cols, m_rows);
  if (p.parts != parts || workspace_of(p, rows, m_rows) > bytes) return 2;
  return launch_plan(p, DenseArgs{x, w, nullptr, y, static_cast<float *>(space), cols, m_rows, rows, cols, rows, p.tiles_m,
                                  p.tiles_n, p.parts, p.steps_per_part}, (hipStream_t)stream);
}
"""


def build(to):
    from georefine_amd import _native
    with tempfile.TemporaryDirectory() as folder:
        source = Path(folder) / "probe.hip"
        source.write_text(PROBE)
        subprocess.run(["hipcc", *_native.HIP_FLAGS, "-shared", "-I", str(ROOT / "include"), "-I", str(SOURCE.parent), str(source),
                        str(SOURCE.parent / "decode_general.hip"), "-o", to], check=True)


def whole(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def drawn_matrix(rng, step):
    cols = max(512, whole(rng, 512, 17408) // step * step)
    return whole(rng, 128, min(17408, 5120 * 17408 // cols)), cols


def best_us(sides, launches, rounds=7):
    """us a call of each side, the sides in turn."""
    import torch
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    best = [math.inf] * len(sides)
    for _ in range(rounds):
        for k, side in enumerate(sides):
            side(0)
            begin.record()
            for i in range(launches):
                side(i)
            end.record()
            end.synchronize()
            best[k] = min(best[k], begin.elapsed_time(end) * 1000 / launches)
    return best


def tilings(probe, out, seed):
    import torch
    lib = ctypes.CDLL(probe)
    u32, ptr = ctypes.c_uint32, ctypes.c_void_p
    lib.probe_dense.argtypes = [u32, u32, ptr, u32, u32, ptr, u32, ptr, ptr, ctypes.c_size_t, ptr]
    rng, launches = random.Random(seed), 12
    products = [(*shape, m) for shape in NAMED for m in (200, 1000)]
    while len(products) < 150:
        rows, cols = drawn_matrix(rng, 8)
        products.append((max(rows, 256), cols, whole(rng, 129, 2048)))
    with open(out, "w", newline="") as file:
        write = csv.writer(file, lineterminator="\n")
        write.writerow(("rows", "cols", "m", "tile", "parts", "us"))
        for count, (rows, cols, m) in enumerate(products):
            ws = [torch.randn(rows, cols, device="cuda").mul_(0.02).bfloat16() for _ in range(3)]
            xs = [torch.randn(m, cols, device="cuda").bfloat16() for _ in range(3)]
            ys = [torch.empty(m, rows, device="cuda", dtype=torch.bfloat16) for _ in range(3)]
            choices = considered(rows, cols, m)
            space = torch.empty(max(p for _, p in choices) * m * (rows + 3), device="cuda")
            first = None
            for tile, parts in choices:
                def launch(i):
                    status = lib.probe_dense(tile, parts, ws[i].data_ptr(), rows, cols, xs[i].data_ptr(), m, ys[i].data_ptr(),
                                             space.data_ptr(), space.numel() * 4, torch.cuda.current_stream().cuda_stream)
                    if status:
                        sys.exit(f"probe: {status} at {rows} x {cols}, {m} rows, tile {tile} in {parts}")
                launch(0)
                torch.cuda.synchronize()
                first = ys[0].float() if first is None else first
                off = (ys[0].float() - first).norm() / first.norm()
                if not off < 5e-3:
                    sys.exit(f"wrong: {rows} x {cols}, {m} rows, tile {tile} in {parts}: {off}")
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph):
                    for i in range(launches):
                        launch(i % 3)
                us = best_us([lambda i: graph.replay()], 2)[0] / launches
                write.writerow((rows, cols, m, tile, parts, round(us, 2)))
                del graph
            file.flush()
            print(count, rows, cols, m, flush=True)


def linear(out, seed):
    import numpy as np
    import torch
    from georefine_amd import _native, _planes, bitexact_context_codec as codec
    from georefine_amd.bitexact_context_gpu import HipContextTensor, dense_linear
    lib = _native.hip()
    _planes.FROM_WEIGHTS = 1 << 40  # what is timed follows the walk's decode: matrices of every size stay frames

    class Asked:
        """The library, with its plan's answer given."""

        def __init__(self, plan):
            self.grf_dense_gemm_plan = plan

        def __getattr__(self, name):
            return getattr(lib, name)

    own, library = Asked(lib.grf_dense_gemm_workspace_bytes), Asked(lambda *sizes: -1)
    rng = random.Random(seed)
    matrices = NAMED + [drawn_matrix(rng, 64 if rng.random() < 0.75 else 16) for _ in range(110)]
    with open(out, "w", newline="") as file:
        write = csv.writer(file, lineterminator="\n")
        write.writerow(("rows", "cols", "m", "us_own", "us_library", "product_own", "product_library"))
        for count, (rows, cols) in enumerate(matrices):
            g = torch.Generator(device="cuda").manual_seed(rows * cols)
            w = torch.randn(rows, cols, device="cuda", generator=g) * 0.02 * torch.exp(0.5 * torch.randn(rows, 1, device="cuda", generator=g))
            w = torch.where(torch.rand(rows, cols, device="cuda", generator=g) < 1e-3, 10.0 * w, w)
            t = HipContextTensor(codec.encode(w.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16), residual="raw6"))
            if t.fused is None:
                continue
            copies = [t, t.clone(), t.clone()]
            dense = [c.decode() for c in copies]
            for m in sorted({whole(rng, 129, 300), whole(rng, 300, 900), whole(rng, 900, 2048)}):
                xs = [torch.randn(m, cols, device="cuda").bfloat16() for _ in range(3)]
                sides = [lambda i, by=by: dense_linear(by, xs[i % 3], copies[i % 3].decode(check=False), None, 0) for by in (own, library)]
                alone = [lambda i, by=by: dense_linear(by, xs[i % 3], dense[i % 3], None, 0) for by in (own, library)]
                us = best_us(sides, 18) + best_us(alone, 18)
                write.writerow((rows, cols, m, *(round(v, 2) for v in us)))
            file.flush()
            print(count, rows, cols, flush=True)


if __name__ == "__main__":
    if sys.argv[1:2] == ["build"]:
        build(sys.argv[2])
    elif sys.argv[1:2] == ["tilings"]:
        tilings(sys.argv[2], sys.argv[3], int(sys.argv[4]) if len(sys.argv) > 4 else 1)
    elif sys.argv[1:2] == ["linear"]:
        linear(sys.argv[2], int(sys.argv[3]) if len(sys.argv) > 3 else 1)
    else:
        sys.exit(__doc__)
