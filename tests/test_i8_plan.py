"""Workspace queries of the int8 GEMM around one and two tiles per CU, in both
tile sizes. The planner divides by the number of tiles past one per CU, which
would end the process, so the queries run in a child process."""

import os
import subprocess
import sys

import pytest

from sparkq import _lib

_CHILD = """
import ctypes, os, sys
lib = ctypes.CDLL(sys.argv[1])
for f in (lib.sparkq_w8a8_workspace_bytes, lib.sparkq_int8_matmul_workspace_bytes):
    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_int64] * 3
edge = int(sys.argv[2])
# tile rows x tile columns of one tile short, exact and one past, with a ragged last tile
for tiles in (255, 256, 257, 511, 512, 513):
    for rows in [r for r in range(2, 33) if tiles % r == 0] + [1]:
        for ragged in (0, 1):
            m, n = edge * rows - ragged, edge * (tiles // rows) - ragged
            if m < 64:
                continue
            for k in (1024, 2560, 4096, 9728):
                lib.sparkq_w8a8_workspace_bytes(m, n, k)
                lib.sparkq_int8_matmul_workspace_bytes(m, n, k)
# ordinary projections at every 64th row
for n in (1024, 2048, 2560, 3584, 4096, 8192, 16384):
    for m in range(64, 4097, 64):
        assert lib.sparkq_w8a8_workspace_bytes(m, n, 4096) > 0
        lib.sparkq_int8_matmul_workspace_bytes(m, n, 4096)
# 256 tiles of 64 x 64: counters, quantized rows and scales, no partial sums
if "SPARKQ_I8_GEMM_SMALL" not in os.environ:
    assert lib.sparkq_w8a8_workspace_bytes(512, 2048, 4096) == 16384 + 512 * 4096 + 512 * 4
print("done")
"""


@pytest.mark.parametrize("edge,small", [(64, "1000000"), (128, "1"), (64, None), (128, None)])
def test_plans_around_one_and_two_tiles_per_cu(edge, small):
    env = dict(os.environ)
    if small is not None:
        env["SPARKQ_I8_GEMM_SMALL"] = small
    r = subprocess.run([sys.executable, "-c", _CHILD, _lib.library_path(), str(edge)], env=env,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "done", (r.returncode, r.stderr)
