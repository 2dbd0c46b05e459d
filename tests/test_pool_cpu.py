"""The library's pool of device blocks, compiled against a stand-in HIP runtime on the
CPU (pool_check.cpp): blocks of several threads, a pointer given back twice, sizes,
and the bounds on what stays idle."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hamiltonian_diagonalization_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pool") / "pool_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-pthread", "-I", CSRC,
                    os.path.join(HERE, "pool_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("name", ["threads", "twice", "sizes", "drain", "bounded", "quarter", "trim"])
def test_pool(check, name):
    assert subprocess.run([check, name], timeout=100).returncode == 0
