"""Where a product of many rows takes the library's matmul and where the framework's own (no GPU)."""
from georefine_amd import _native


def test_plan_by_sizes():
    plan = _native.hip().grf_dense_gemm_plan
    need = _native.hip().grf_dense_gemm_workspace_bytes
    assert plan(5120, 17408, 1000) == need(5120, 17408, 1000) > 0  # long rows: cut along K
    assert plan(5120, 17408, 2048) == -1 and plan(17408, 5120, 1000) == -1 and plan(1024, 4096, 1536) == -1  # outputs that fill the GPU
    assert plan(640, 512, 150) >= 0  # short work
    for refused in ((0, 512, 150), (640, 0, 150), (640, 512, 0), (640, 516, 150), (640, (1 << 21) + 8, 150), (1 << 24, 512, 150)):
        assert plan(*refused) == -1 and need(*refused) == 0
    for rows in (1, 63, 300, 5120, 17408):
        for cols in (8, 72, 4096, 17408):
            for m in (129, 300, 1000, 4096):
                size = need(rows, cols, m)
                pitch = (rows + 3) // 4 * 4
                assert size % (4 * m * pitch) == 0 and size <= 64 * 4 * m * pitch
