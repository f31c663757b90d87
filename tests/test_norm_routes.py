"""The rules that choose between the fused norms' kernels (csrc/norm_route.h,
plain host C++), built with g++ and read on the CPU."""
import ctypes
import os
import shutil
import subprocess

import pytest

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "minimax-h3-multi-dgx-spark_amd", "csrc", "norm_route.h")


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    src, lib = str(d / "routes.cpp"), str(d / "routes.so")
    with open(src, "w") as f:
        f.write(f'#include "{HEADER}"\n'
                'extern "C" int norm_rows(int gate, int quant, int64_t S, int64_t N, int64_t R) '
                '{ return h3mi::norm_rows_suit(gate, quant, S, N, R); }\n'
                'extern "C" int gate_rows(int64_t S, int64_t N, int64_t R) { return h3mi::gate_rows_suit(S, N, R); }\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", lib, src], check=True)
    so = ctypes.CDLL(lib)
    i = ctypes.c_int64
    so.norm_rows.argtypes = [ctypes.c_int, ctypes.c_int, i, i, i]
    so.gate_rows.argtypes = [i, i, i]
    ops = {"norm_mod": (0, 0), "norm_mod_q": (0, 1), "gate_norm_mod_": (1, 0), "gate_norm_mod_q_": (1, 1)}
    return lambda op, S, N, R: bool(so.gate_rows(S, N, R) if op == "gate_" else so.norm_rows(*ops[op], S, N, R))


OPS = ["norm_mod", "norm_mod_q", "gate_norm_mod_", "gate_norm_mod_q_", "gate_"]


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("N", [8, 64, 1024, 2048, 3072, 8192])
@pytest.mark.parametrize("R", [1, 2, 5])
def test_no_workgroup_per_row_past_the_launch_limit(routes, op, N, R):
    """2^24 workgroups of 256 threads are 2^32 threads, which HIP refuses."""
    for S in (1 << 24, (1 << 24) + 1, (1 << 31) - 1):
        assert not routes(op, S, N, R)


@pytest.mark.parametrize("op,S,N,R,rows", [
    # (route of the faster side as measured: rows = one row per workgroup)
    ("norm_mod", 4800, 2048, 1, True), ("norm_mod", 9600, 512, 1, False), ("norm_mod", 9600, 3072, 1, False),
    ("norm_mod", 38400, 512, 2, True), ("norm_mod", 38400, 5376, 2, False), ("norm_mod", 38400, 5120, 5, True),
    ("norm_mod_q", 3600, 5376, 1, True), ("norm_mod_q", 4600, 5376, 1, False), ("norm_mod_q", 2400, 8192, 1, True),
    ("norm_mod_q", 4800, 512, 2, True), ("norm_mod_q", 9600, 512, 2, False), ("norm_mod_q", 38400, 128, 5, False),
    ("norm_mod_q", 19200, 1024, 2, False), ("norm_mod_q", 200000, 64, 2, False), ("norm_mod_q", 14400, 2048, 2, True),
    ("norm_mod_q", 7200, 5376, 2, False), ("norm_mod_q", 3000, 8192, 5, True),
    ("gate_norm_mod_", 38400, 1024, 1, True), ("gate_norm_mod_", 38400, 1536, 1, False),
    ("gate_norm_mod_", 4800, 1536, 1, True), ("gate_norm_mod_", 28800, 1032, 2, False),
    ("gate_norm_mod_", 19200, 2560, 2, False), ("gate_norm_mod_", 7200, 2560, 2, True),
    ("gate_norm_mod_", 38400, 5376, 2, True), ("gate_norm_mod_", 38400, 512, 2, True),
    ("gate_norm_mod_q_", 19200, 3072, 2, False), ("gate_norm_mod_q_", 9600, 3072, 2, True),
    ("gate_norm_mod_q_", 28800, 3584, 2, False), ("gate_norm_mod_q_", 38400, 512, 2, True),
    ("gate_norm_mod_q_", 19200, 5376, 5, True), ("gate_norm_mod_q_", 9600, 512, 1, False),
    ("gate_", 38400, 4096, 1, True), ("gate_", 19200, 5376, 1, False), ("gate_", 38400, 5376, 2, True),
])
def test_route_of_the_faster_side(routes, op, S, N, R, rows):
    assert routes(op, S, N, R) == rows


def test_the_gpu_tests_of_the_streams_reach_them(routes):
    import test_gpu_norm_routes as t
    for S, N, R, ops in t.STREAMS:
        for op in ops:
            assert not routes(op, S, N, R), (op, S, N, R)
            assert routes(op, 700, N, R)  # the calls they are held against
