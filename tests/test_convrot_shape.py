"""The rule that picks the ConvRot quantizer's waves per row and passes per
wave (csrc/convrot_shape.h, plain host C++), built with g++ and read on the CPU."""
import ctypes
import os
import shutil
import subprocess

import pytest

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "minimax-h3-multi-dgx-spark_amd", "csrc", "convrot_shape.h")


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    d = tmp_path_factory.mktemp("shape")
    src, lib = str(d / "shape.cpp"), str(d / "shape.so")
    with open(src, "w") as f:
        f.write(f'#include "{HEADER}"\n'
                'extern "C" int shape(int chunks, int swiglu, int64_t rows) '
                '{ int w = 0, p = 0; h3mi::convrot_shape(chunks, swiglu, rows, 256, &w, &p); return 100 * w + p; }\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", lib, src], check=True)
    so = ctypes.CDLL(lib)
    so.shape.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64]
    return lambda K, swiglu, rows: divmod(so.shape(-(-K // 1024), swiglu, rows), 100)


@pytest.mark.parametrize("K,swiglu,rows,want", [
    # (waves per row, passes) of the faster shape as measured
    (5376, 0, 37, (8, 1)), (5376, 0, 1536, (8, 1)), (5376, 0, 1537, (2, 3)), (3072, 0, 512, (4, 1)),
    (9216, 0, 37, (4, 3)), (12288, 0, 1024, (4, 3)), (14336, 0, 37, (8, 2)), (24832, 0, 37, (8, 4)),
    (5376, 1, 256, (8, 1)), (5376, 1, 257, (2, 3)), (6144, 1, 384, (2, 3)), (4608, 1, 384, (2, 3)),
    (7168, 1, 384, (8, 1)), (3072, 1, 384, (4, 1)), (9216, 1, 96, (4, 3)), (12288, 1, 384, (4, 3)),
    (14336, 1, 384, (8, 2)), (14336, 1, 385, (4, 4)),
])
def test_shape_as_measured(shape, K, swiglu, rows, want):
    assert shape(K, swiglu, rows) == want


@pytest.mark.parametrize("swiglu", [0, 1])
@pytest.mark.parametrize("rows", [1, 300, 19200])
def test_every_row_is_covered(shape, swiglu, rows):
    for K in range(256, 32769, 256):
        w, p = shape(K, swiglu, rows)
        assert w in (1, 2, 4, 8) and 1 <= p <= 8 and w * p * 1024 >= K
