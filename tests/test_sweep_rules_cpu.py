"""The host rules of the SpMM sweep kernel (library_amd/csrc/asx_internal.hpp) over sizes drawn at random, tests/cxx/sweep_rules.cpp."""
import os
import subprocess

from library_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rules(tmp_path):
    exe = str(tmp_path / "sweep_rules")
    flags = [f for f in build.HIP_FLAGS if not f.startswith("-Rpass") and f != "-O3"]
    subprocess.run([build.HIPCC, "-x", "hip", *flags, "-O1", os.path.join(HERE, "cxx", "sweep_rules.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
