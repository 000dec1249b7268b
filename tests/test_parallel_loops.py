"""The layout builders' threaded loops (csrc/parallel.h) on the host: every index once, exceptions carried to the caller,
threads that cannot be started replaced by the caller."""

import os
import subprocess

import pytest

from conftest import PKG, ROOT


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("cpp") / "parallel_loops")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-Wall", "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "parallel_loops.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("what", ["ranges", "throws", "no_threads"])
def test_parallel_loops(program, what):
    assert subprocess.run([program, what], timeout=60).returncode == 0
