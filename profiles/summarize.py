"""Profiles bench.py's workloads and those of prompts.py with rocprofv3 and writes the summaries that lie beside this file.

    python3 profiles/summarize.py OUT [NAME ...]

NAME: a key of WORKLOADS (default: all).  For each, one kernel trace and five counter runs (a run holds
so many counters of a block), then OUT/NAME.txt, a table for readers, and OUT/NAME_traffic.json, which
bench.py reads while the kernel sources are the ones recorded in it.  The whole stack is traced only.

What the derived lines say (MI355X: 8 XCDs, 256 compute units, 1024 SIMDs):
  cycles of a launch     GRBM_GUI_ACTIVE / 8, since every XCD counts its own
  VALU busy              4 SQ_ACTIVE_INST_VALU / (1024 cycles): the counter is in quad-cycles, summed over SIMDs
  LDS busy               SQ_LDS_IDX_ACTIVE / (256 cycles): cycles the units' LDS pipes worked on indexed accesses
                         (SQ_ACTIVE_INST_LDS counts the issue of the instructions only, and says next to
                         nothing about the pipe), with the share SQ_LDS_BANK_CONFLICT of them
  matrix cores busy      SQ_VALU_MFMA_BUSY_CYCLES / (1024 cycles)
  per wave step          totals / (weights / 64), of the walk: a wave step is one symbol for each of a wave's 64 lanes
"""
import collections
import csv
import glob
import json
import os
import statistics
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402

MLP = "Qwen-27B-like MLP (gate, up: 17408x5120; down: 5120x17408), MI355X (gfx950)"
MATRIX = 5120 * 17408
# title, the program's options (the program first where it is not bench.py), {kernel: weights a launch walks, or 0}, what the traffic
# record is called
WORKLOADS = {
    "planes_m1_gate_up": (
        "Product of planes, one row, gate and up (17408x5120 each) in one grouped launch, MI355X (gfx950)",
        ["--only", "gate,up"], {"planes_product_kernel": 0}, "gate and up in one launch, batch 1"),
    "planes_m64_gate_up": (
        "Product of planes, 64 rows, gate and up (17408x5120 each) in one grouped launch, MI355X (gfx950)",
        ["--batch", "64", "--only", "gate,up"], {"planes_batch_kernel": 0, "planes_sum_kernel": 0}, "gate and up in one launch, batch 64"),
    "planes_decode_qwen27b_mlp": (
        f"Planes to dense BF16 (decode()), {MLP}\none step = three launches",
        ["--workload", "decode"], {"planes_decode_kernel": 0}, "Qwen-27B-like MLP decode"),
    "planes_ppcx_m1_5120x17408": (
        "Product of a predictive (PPCX) weight held as planes, 5120x17408, batch 1, MI355X (gfx950)",
        ["--workload", "ppcx", "--batch", "1"], {"planes_product_kernel": 0, "planes_sum_kernel": 0}, "PPCX 5120x17408 batch 1"),
    "planes_ppcx_m96_5120x17408": (
        "Product of a predictive (PPCX) weight held as planes, 5120x17408, 96 rows, MI355X (gfx950)",
        ["--workload", "ppcx", "--batch", "96"], {"planes_batch_kernel": 0, "planes_sum_kernel": 0}, "PPCX 5120x17408 batch 96"),
    "planes_prompt_m1000_5120x17408": (
        "A prompt of 1000 rows through 5120x17408 held as planes, MI355X (gfx950)",
        ["profiles/prompts.py", "prompt"], {"planes_prompt_kernel": 0, "dense_sum_kernel": 0}, "prompt of 1000 rows, 5120x17408"),
    "planes_lookup_777_of_8192x5120": (
        "An embedding lookup, 777 rows of 8192x5120 held as planes, MI355X (gfx950)",
        ["profiles/prompts.py", "lookup"], {"planes_gather_kernel": 0}, "lookup of 777 rows, 8192x5120"),
    "planes_m64_stack_64_layers": (
        "Whole stack at the 27B model's shapes: 64 layers (48 with gated-delta-net projections, 16 with attention q/k/v/o) x "
        "(projections, gate, up, down) + embedding and head (248320x5120), batch 64, held as planes, MI355X (gfx950)",
        ["--workload", "stack", "--steps", "3", "--warmup", "1"], {}, ""),
    # the walk, which small matrices and frames of few exponents take, at the same sizes
    "fused_gemv_m1_qwen27b_mlp": (
        f"Fused decode-GEMV (wave units), batch 1, {MLP}\n"
        "one step = gate and up in one grouped launch (they take the same activations) + down in a launch of its own",
        ["--walked"], {"fused_wave_group_kernel": 2 * MATRIX, "fused_wave_kernel": MATRIX}, "Qwen-27B-like MLP batch 1"),
    "fused_gemm_m64_qwen27b_mlp": (
        f"Fused decode-GEMM (matrix cores), batch 64, {MLP}\n"
        "one step = gate and up in one grouped launch + down cut in three along K",
        ["--walked", "--batch", "64"], {"fused_gemm_group_kernel": 2 * MATRIX, "fused_gemm_kernel": MATRIX}, "Qwen-27B-like MLP batch 64"),
    "fused_store_decode_qwen27b_mlp": (
        f"Fused decode to dense BF16 (store sink over wave units), {MLP}\none step = three launches",
        ["--walked", "--workload", "decode"], {"fused_wave_store_kernel": MATRIX}, "Qwen-27B-like MLP decode"),
    "ppcx_gemv_m1_5120x17408": (
        "Fused decode-GEMV of a predictive (PPCX) weight, 5120x17408, batch 1, MI355X (gfx950)",
        ["--walked", "--workload", "ppcx", "--batch", "1"], {"fused_wave_kernel": MATRIX}, "PPCX 5120x17408 batch 1"),
    "ppcx_gemm_m96_5120x17408": (
        "Fused decode-GEMM of a predictive (PPCX) weight, 5120x17408, 96 rows, MI355X (gfx950)",
        ["--walked", "--workload", "ppcx", "--batch", "96"],
        {"fused_gemm_wide_kernel": MATRIX, "pack_activations_kernel": 0, "gemm_sum_parts_kernel": 0}, "PPCX 5120x17408 batch 96"),
    "prompt_m1000_5120x17408": (
        "A prompt of 1000 rows through 5120x17408: fused decode to dense BF16, then the product over it, MI355X (gfx950)",
        ["profiles/prompts.py", "prompt", "--walked"], {"dense_gemm_kernel": 0, "dense_sum_kernel": 0, "fused_wave_store_kernel": MATRIX},
        "prompt of 1000 rows, 5120x17408"),
    "lookup_777_of_8192x5120": (
        "An embedding lookup, 777 rows of 8192x5120, MI355X (gfx950)",
        ["profiles/prompts.py", "lookup", "--walked"], {"fused_gather_kernel": 777 * 5120}, "lookup of 777 rows, 8192x5120"),
    "fused_gemm_m64_stack_64_layers": (
        "Whole stack at the 27B model's shapes: 64 layers (48 with gated-delta-net projections, 16 with attention q/k/v/o) x "
        "(projections, gate, up, down) + embedding and head (248320x5120), batch 64, MI355X (gfx950)",
        ["--walked", "--workload", "stack", "--steps", "3", "--warmup", "1"], {}, ""),
}
COUNTERS = (
    "SQ_WAVES SQ_INSTS_VALU SQ_INSTS_LDS SQ_INSTS_SALU SQ_ACTIVE_INST_VALU SQ_ACTIVE_INST_LDS SQ_BUSY_CU_CYCLES SQ_WAVE_CYCLES",
    "SQ_LDS_BANK_CONFLICT SQ_LDS_IDX_ACTIVE SQ_LDS_ADDR_CONFLICT SQ_WAIT_INST_LDS SQ_WAIT_INST_ANY SQ_INSTS_VMEM_RD "
    "SQ_LDS_UNALIGNED_STALL GRBM_GUI_ACTIVE",
    "SQ_VALU_MFMA_BUSY_CYCLES GRBM_GUI_ACTIVE", "FETCH_SIZE", "WRITE_SIZE")
COPY_BYTES = 128 << 20  # of bench.py's calibration copy, read once and written once
RUN_SECONDS = 150


def short(kernel):
    return kernel.replace("(anonymous namespace)", "").split("(")[0].split("<")[0].split("::")[-1].replace("void ", "").strip()


def command(arguments):
    if arguments[:1] and arguments[0].endswith(".py"):
        return [arguments[0], "--calibrate-copy", *arguments[1:]]
    return ["bench.py", "--no-cpu-baseline", "--no-extras", "--calibrate-copy", *arguments]


def profiled(scratch, tag, options, arguments):
    """One profiled run of the workload's program; the directory with its CSV files."""
    into = os.path.join(scratch, tag)
    program, *rest = command(arguments)
    done = subprocess.run(
        ["timeout", "-s", "KILL", str(RUN_SECONDS), "rocprofv3", *options, "-d", into, "-o", "r", "-f", "csv", "--", "python3",
         os.path.join(ROOT, program), *rest],
        cwd=scratch, env=dict(os.environ, TMPDIR=scratch), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    finished = any(line.startswith('{"metric"') for line in done.stdout.splitlines())
    print(tag, done.returncode, flush=True)
    if not finished:
        sys.exit(done.stdout[-2000:])
    return into


def counters(directory):
    """{kernel: {counter: [value of every dispatch]}}"""
    found = collections.defaultdict(lambda: collections.defaultdict(list))
    for path in glob.glob(directory + "/**/*counter_collection.csv", recursive=True):
        total, kernel = collections.defaultdict(float), {}
        for row in csv.DictReader(open(path)):
            total[row["Dispatch_Id"], row["Counter_Name"]] += float(row["Counter_Value"])
            kernel[row["Dispatch_Id"]] = row["Kernel_Name"]
        for (dispatch, counter), value in total.items():
            found[kernel[dispatch]][counter].append(value)
    return found


def derived(m, weights):
    """The lines of one kernel's mean counters ``m`` that the totals do not show."""
    cycles = m["GRBM_GUI_ACTIVE"] / 8
    lines = [f"  -> {m['SQ_WAVES']:.0f} waves; VALU instructions per wave {m['SQ_INSTS_VALU'] / m['SQ_WAVES']:.0f}, LDS instructions "
             f"per wave {m['SQ_INSTS_LDS'] / m['SQ_WAVES']:.0f}; cycles of the launch {cycles:.0f} (GRBM_GUI_ACTIVE / 8 XCDs)"]
    if weights:
        steps = weights / 64
        lines.append(f"  -> per wave and symbol step, everything outside the step loop included: {m['SQ_INSTS_VALU'] / steps:.1f} VALU, "
                     f"{m['SQ_INSTS_LDS'] / steps:.2f} LDS, {m['SQ_INSTS_SALU'] / steps:.1f} SALU, {m['SQ_INSTS_VMEM_RD'] / steps:.3f} "
                     f"vector-memory read instructions; {m['SQ_LDS_IDX_ACTIVE'] / steps:.1f} LDS cycles")
    conflicts = m["SQ_LDS_BANK_CONFLICT"] / m["SQ_LDS_IDX_ACTIVE"] if m["SQ_LDS_IDX_ACTIVE"] else 0.0
    lines.append(f"  -> VALU busy {100 * 4 * m['SQ_ACTIVE_INST_VALU'] / (1024 * cycles):.1f} % of the launch's cycles (SQ_ACTIVE_INST_VALU "
                 f"counts quad-cycles, 1024 SIMDs); LDS busy {100 * m['SQ_LDS_IDX_ACTIVE'] / (256 * cycles):.1f} % (SQ_LDS_IDX_ACTIVE, 256 "
                 f"units), of which bank conflicts {100 * conflicts:.1f} %; waves waiting on anything "
                 f"{100 * m['SQ_WAIT_INST_ANY'] / m['SQ_WAVE_CYCLES']:.1f} % of their cycles")
    if m["SQ_VALU_MFMA_BUSY_CYCLES"]:
        lines.append(f"  -> matrix cores busy {100 * m['SQ_VALU_MFMA_BUSY_CYCLES'] / (1024 * cycles):.1f} % of the launch's cycles")
    return lines


def summarize(name, out, scratch):
    title, arguments, kernels, workload = WORKLOADS[name]
    fewer = [*arguments, "--steps", "20", "--warmup", "10"]
    times = collections.defaultdict(list)
    for path in glob.glob(profiled(scratch, name + "_trace", ["--kernel-trace", "--stats"], arguments) + "/**/*kernel_trace.csv",
                          recursive=True):
        for row in csv.DictReader(open(path)):
            start, end = int(row["Start_Timestamp"]), int(row["End_Timestamp"])
            times[row["Kernel_Name"]].append((start, (end - start) / 1e3))
    text = [title, "rocprofv3 summaries (profiles/summarize.py) of",
            "  T = python3 " + " ".join(command(arguments)) + "      (its own warm-up and timed steps)",
            *(["  B = T --steps 20 --warmup 10      (counter runs serialise the kernels: fewer steps)"] if kernels else []),
            *(["  (eager calls;"] if command(arguments)[0] != "bench.py" else
              ["  (warm-up launches are eager; the timed ones are replays of HIP graphs, launched back to back as in the bench line;"]),
            "   steps and launches take several device copies of the matrices in turn, so no matrix is found in the last-level cache;",
            "   --calibrate-copy adds one plain copy kernel of known size, read by the traffic counters of the runs that take them)",
            "  rocprofv3 --kernel-trace --stats -- T", *(f"  rocprofv3 --pmc {c} -- B" for c in COUNTERS if kernels), "", "kernel trace:"]
    whole = sum(t for launches in times.values() for _, t in launches)
    for kernel, launches in sorted(times.items(), key=lambda item: -sum(t for _, t in item[1]))[:8]:
        total = sum(t for _, t in launches)
        text.append(f"  {kernel[:96]:<96} calls {len(launches):4d} total {total:10.1f} us  avg {total / len(launches):8.2f} us  "
                    f"{100 * total / whole:5.1f}%")
    for kernel in kernels:
        us = [t for _, t in sorted(x for k, launches in times.items() if short(k) == kernel for x in launches)]
        text.append(f"  {kernel}: {len(us)} launches, mean {statistics.mean(us):.2f} us, median {statistics.median(us):.2f} us, mean of "
                    f"the later half {statistics.mean(us[len(us) // 2:]):.2f} us, fastest {min(us):.2f} us")
    sources = bench.kernel_sources_sha256()
    if not kernels:
        with open(os.path.join(out, name + ".txt"), "w") as f:
            f.write("\n".join([*text, "", "kernel sources sha256 " + sources]) + "\n")
        return
    values, copy = collections.defaultdict(lambda: collections.defaultdict(list)), collections.defaultdict(list)
    for i, names in enumerate(COUNTERS):
        for kernel, found in counters(profiled(scratch, f"{name}_counters{i}", ["--pmc", *names.split()], fewer)).items():
            for counter, of in found.items():
                if short(kernel) in kernels:
                    values[short(kernel)][counter] += of
                elif "CUDAFunctorOnSelf_add<int>" in kernel:  # the calibration copy
                    copy[counter] += of
    fetch_scale, write_scale = (COPY_BYTES / (statistics.mean(copy[c]) * 1024) for c in ("FETCH_SIZE", "WRITE_SIZE"))
    traffic = {}
    for kernel, weights in kernels.items():
        m = {counter: statistics.mean(of) for counter, of in values[kernel].items()}
        fetched, written = m["FETCH_SIZE"] * 1024 * fetch_scale, m["WRITE_SIZE"] * 1024 * write_scale
        traffic[kernel] = fetched + written
        text += ["", f"counters, mean per launch of {kernel} (whole GPU):", *(f"  {c:<30} {m[c]:14.1f}" for c in sorted(m)),
                 f"  -> HBM-side traffic per launch: fetch {fetched / 1e6:.1f} MB + write {written / 1e6:.2f} MB = "
                 f"{(fetched + written) / 1e6:.1f} MB", *derived(m, weights)]
    text += ["", f"traffic scale from the copy kernel: FETCH_SIZE x {fetch_scale:.4f}, WRITE_SIZE x {write_scale:.4f} KiB",
             "kernel sources sha256 " + sources]
    if workload.startswith("PPCX"):  # (a product may be several launches)
        traffic = {"product": sum(traffic.values()), **traffic}
    with open(os.path.join(out, name + ".txt"), "w") as f:
        f.write("\n".join(text) + "\n")
    with open(os.path.join(out, name + "_traffic.json"), "w") as f:
        f.write(json.dumps({"workload": workload, "traffic_bytes_per_launch": traffic, "fetch_scale": fetch_scale,
                            "write_scale": write_scale, "kernel_sources_sha256": sources}) + "\n")


if __name__ == "__main__":
    if len(sys.argv) < 2 or any(n not in WORKLOADS for n in sys.argv[2:]):
        sys.exit(__doc__)
    os.makedirs(sys.argv[1], exist_ok=True)
    with tempfile.TemporaryDirectory() as scratch_dir:
        for wanted in sys.argv[2:] or WORKLOADS:
            summarize(wanted, os.path.abspath(sys.argv[1]), scratch_dir)
            print(wanted, "done", flush=True)
