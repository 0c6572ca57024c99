"""norm_gate_workspace_bytes (host logic; 256 CUs assumed without a device): one row of partial column sums per workgroup of the
backward pass, whose workgroups have 1024 threads with 16-bit elements - but 256 where rows of one or two wavefronts are so
few that each workgroup has a CU and one group of rows."""
from lightning_attn.ops.hip import _lib


def test_workgroups_of_the_backward_pass():
    L = _lib.lib()
    groups = lambda rows, cols, dtype: L.norm_gate_workspace_bytes(rows, cols, dtype) / (2 * cols * 4)  # noqa: E731
    for dtype in (0, 1):
        for cols, per256 in ((64, 4), (512, 4), (520, 2), (1024, 2)):
            assert groups(1, cols, dtype) == 1 and groups(per256 + 1, cols, dtype) == 2
            assert groups(256 * per256, cols, dtype) == 256
            assert groups(256 * per256 + 1, cols, dtype) == 64 + 1  # four times as many rows to a workgroup
            assert groups(10 ** 6, cols, dtype) == 256
        assert groups(200, 2048, dtype) == 50 and groups(200, 8192, dtype) == 200
    assert groups(1024, 64, 2) == 256 and groups(10 ** 6, 64, 2) == 1024


def test_workspace_of_many_short_rows_is_enough_for_fewer():
    """(rows that share a wavefront leave fewer partial sums than the fewer rows which get a wavefront each)"""
    L = _lib.lib()
    for dtype, most in ((0, 256), (1, 256), (2, 1024)):
        for cols in (64, 128, 200, 256) if dtype < 2 else (32, 64, 100, 128):
            for rows in (4096, 4097, 5000, 8192, 8193, 16385, 10 ** 6):
                assert L.norm_gate_workspace_bytes(rows, cols, dtype) == most * 2 * cols * 4, (rows, cols, dtype)
