"""State downloads (sfv_transfer.hip, built for the CPU over a stand-in for the
HIP runtime): the bytes of copies around the staged size, destinations that the
runtime knows, and what the staging memory and streams of one copy leave
behind."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "volumefluxes.jl_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("transfer") / "transfer")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(HERE, "stub_hip"), "-I", CSRC,
                    os.path.join(HERE, "stub_hip", "transfer_main.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["pageable", "device_destination", "pinned_destination", "callers_stream",
                                      "one_after_the_other", "many_at_once", "failing"])
def test_copy_to_host(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
