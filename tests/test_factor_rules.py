"""Launch rules of the device factorisation (linearalgebra_amd/csrc/
host_algos.hpp), called on the CPU (tests/cpp/factor_capi.cpp, built here
with g++)."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

from helpers import ROOT


@pytest.fixture(scope="module")
def fac(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    so = str(tmp_path_factory.mktemp("factor") / "libfactor.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "linearalgebra_amd", "csrc"), "-o", so,
                    os.path.join(ROOT, "tests", "cpp", "factor_capi.cpp")],
                   check=True, timeout=300)
    return C.CDLL(so)


@pytest.mark.parametrize("chunks,levels,wgs", [
    (1, 1, 1), (63, 1, 63), (1000, 1000, 64), (1000, 100, 120), (5000, 10, 1024),
    (178956970, 1, 1024), (178956971, 1, 1024), (2 ** 31 - 1, 1, 1024),
    (2 ** 31 - 1, 2 ** 28, 95), (2 ** 31 - 1, 2 ** 31 - 1, 64)])
def test_workgroups(fac, chunks, levels, wgs):
    """12 levels of chunks, at least 64 and at most 1024 workgroups, never
    more than there are chunks: up to the largest number of chunks."""
    assert fac.fac_workgroups(chunks, levels) == wgs


@pytest.mark.parametrize("rows,levels,lanes,eliminations,one", [
    (260, 259, 64, 8190, 1),              # banded: a chain of rows
    (4096, 127, 8, 8064, 1),              # 64^2 5-point cells
    (110592, 612, 64, 3300000, 1),        # 48^3 27-point ILU(1)
    (2097152, 2, 8, 6242304, 1),          # 128^3 7-point cells by colour
    (1000000, 1, 4, 0, 1),                # a diagonal matrix
    (200000, 40, 64, 3900000, 1),         # dense blocks of 40 rows
    (500000, 17, 32, 1000000, 0),         # random graph, mean degree 4
    (500000, 12, 16, 500000, 0),          # mean degree 2, rows up to 13
    (500000, 26, 32, 2000000, 1),         # mean degree 8
    (2000000, 12, 16, 2000000, 0),        # mean degree 2, rows up to 14
    (20000, 2, 64, 59, 0),                # a diagonal and one row of 60
    (2000, 2, 64, 59, 1),
    (0, 1, 4, 0, 1),
    (2 ** 31 - 1, 3, 64, 2 ** 31 - 1, 0)])
def test_one_launch(fac, rows, levels, lanes, eliminations, one):
    """The faster form by measurement, on both sides of the line."""
    assert fac.fac_one_launch(C.c_longlong(rows), C.c_longlong(levels), lanes,
                              C.c_longlong(eliminations)) == one
