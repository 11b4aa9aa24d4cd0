"""Launch rules of the device factorisation and the tiled triangular solve
(linearalgebra_amd/csrc/host_algos.hpp), called on the CPU (tests/cpp/
launch_rules_capi.cpp, built here with g++)."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

from helpers import ROOT


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    so = str(tmp_path_factory.mktemp("rules") / "librules.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "linearalgebra_amd", "csrc"), "-o", so,
                    os.path.join(ROOT, "tests", "cpp", "launch_rules_capi.cpp")],
                   check=True, timeout=300)
    return C.CDLL(so)


@pytest.mark.parametrize("chunks,levels,wgs", [
    (1, 1, 1), (63, 1, 63), (1000, 1000, 64), (1000, 100, 120), (5000, 10, 1024),
    (178956970, 1, 1024), (178956971, 1, 1024), (2 ** 31 - 1, 1, 1024),
    (2 ** 31 - 1, 2 ** 28, 95), (2 ** 31 - 1, 2 ** 31 - 1, 64)])
def test_factor_workgroups(rules, chunks, levels, wgs):
    """12 levels of chunks, at least 64 and at most 1024 workgroups, never
    more than there are chunks: up to the largest number of chunks."""
    assert rules.fac_workgroups(chunks, levels) == wgs


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
def test_factor_one_launch(rules, rows, levels, lanes, eliminations, one):
    """The faster form by measurement, on both sides of the line."""
    assert rules.fac_one_launch(C.c_longlong(rows), C.c_longlong(levels), lanes,
                              C.c_longlong(eliminations)) == one


@pytest.mark.parametrize("active,record,touch", [
    (46, 5632, 1), (47, 5632, 0),      # eight FP64 values a lane: 8.29 / 8.47 MB
    (78, 3328, 1), (79, 3328, 0),      # eight FP32 values
    (73, 3584, 1), (74, 3584, 0),      # four FP64 values
    (128, 2048, 1), (129, 2048, 0)])   # two FP64 values: 2^23 bytes exactly
def test_tile_touch(rules, active, record, touch):
    """Records between a touch and its use: four blocks of eight groups of
    every active tile, however long the plan's rings are; 2^23 bytes at most."""
    assert 32 * active * record <= 2 ** 23 if touch else 32 * active * record > 2 ** 23
    levels = 1345
    groups = C.c_longlong((active - 1) * levels + 7)
    assert rules.tri_touch(groups, C.c_longlong(levels), C.c_longlong(record)) == touch
