"""The pool of device memory (library_amd/csrc/asx_pool.cpp), linked with a HIP that tests/cxx/pool_check.cpp plays on the host."""
import os
import subprocess

import pytest

from library_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def pool_check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("pool") / "pool_check"
    subprocess.run(["g++", *build.CXX_FLAGS, os.path.join(HERE, "cxx", "pool_check.cpp"), os.path.join(build.CSRC, "asx_pool.cpp"),
                    "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("case", ["kept", "refused_wait_of_a_plan", "refused_wait_of_a_call", "relaxed_capture", "device_reset"])
def test_pool(pool_check, case):
    run = subprocess.run([pool_check, case], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
