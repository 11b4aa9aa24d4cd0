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
