"""bench.py's command line on a machine without a GPU: what it refuses, and the helpers that
need no device."""
import json
import subprocess
import sys
import types
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def test_more_than_one_gpu_is_refused():
    run = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert run.returncode != 0
    assert "one GPU" in run.stderr and not run.stdout.strip()


def test_recorded_traffic_is_withheld_for_other_kernel_sources(monkeypatch):
    sys.path.insert(0, str(ROOT))
    import bench
    name = "grf::fused_wave_group_kernel<grf::SegmentWalkT<false>, 1, 1>"
    record = json.loads((ROOT / "profiles" / "fused_gemv_m1_qwen27b_mlp_traffic.json").read_text())
    monkeypatch.setattr(bench, "kernel_sources_sha256", lambda: record["kernel_sources_sha256"])
    figure, source = bench.recorded_traffic(False, 1, name)
    assert figure == record["traffic_bytes_per_launch"]["fused_wave_group_kernel"] and "recorded" in source
    monkeypatch.setattr(bench, "kernel_sources_sha256", lambda: "0" * 64)
    figure, source = bench.recorded_traffic(False, 1, name)
    assert figure is None and "other kernel sources" in source
    assert bench.recorded_traffic(False, 7, name)[0] is None  # no counter record for that batch
    assert "planes_ppcx_m96_5120x17408" in bench.recorded_traffic(False, 96, "planes_batch_kernel", prefix="ppcx")[1]
    assert "no counter record" in bench.recorded_traffic(False, 32, "planes_product_kernel or planes_batch_kernel")[1]


@pytest.mark.parametrize("profile,decode_only,m,grouped", [
    ("fused_gemv_m1_qwen27b_mlp", False, 1, True), ("fused_gemv_m1_qwen27b_mlp", False, 1, False),
    ("fused_gemm_m64_qwen27b_mlp", False, 64, True), ("fused_gemm_m64_qwen27b_mlp", False, 64, False),
    ("fused_store_decode_qwen27b_mlp", True, 1, False), ("planes_m1_gate_up", False, 1, True), ("planes_m64_gate_up", False, 64, True),
    ("planes_decode_qwen27b_mlp", True, 0, False), ("planes_ppcx_m1_5120x17408", False, 1, False),
    ("planes_ppcx_m96_5120x17408", False, 96, False)])
def test_kernels_it_names_are_the_ones_that_were_profiled(profile, decode_only, m, grouped):
    sys.path.insert(0, str(ROOT))
    import bench
    name = bench.kernel_name(decode_only, m, grouped, planes=profile.startswith("planes"))
    assert name.split(", MT")[0].rstrip(">") in (ROOT / "profiles" / f"{profile}.txt").read_text()
    record = json.loads((ROOT / "profiles" / f"{profile}_traffic.json").read_text())
    assert name.split("<")[0].split("::")[-1] in record["traffic_bytes_per_launch"]


class _Held:
    """A predictive tensor that is held as planes, of which nothing of the walk may be asked."""
    shape, fusable, host_bytes = (5120, 17408), True, 7
    _planes = types.SimpleNamespace(nbytes=128000000, splits=12)
    resident_bytes = 128000004

    def __getattr__(self, name):
        raise AssertionError(f"{name} was asked for")


def test_predictive_products_are_counted_in_the_form_they_are_held_in():
    sys.path.insert(0, str(ROOT))
    import bench
    for m, kernel in ((1, "planes_product_kernel"), (96, "planes_batch_kernel")):
        assert bench.predictive_product(_Held(), m) == (128000000 + m * 2 * (5120 + 17408), kernel)
