"""State uploads and downloads where the device or a copy refuses, on a runtime of host memory (transfers/transfers.cpp):
the C ABI's own source, compiled for the host."""
import os
import subprocess

import pytest

from rsim import build as rb

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("transfers") / "transfers")
    rocm = os.path.dirname(os.path.dirname(rb._hipcc()))
    cmd = ["g++"] + rb.COMMON + ["-O1", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(rocm, "include"),
                                 os.path.join(HERE, "transfers", "transfers.cpp"), os.path.join(rb.CSRC, "host", "rsim.cpp"),
                                 "-Wl,--unresolved-symbols=ignore-all", "-o", out]  # the launchers that no case calls
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-4000:]
    return out


@pytest.mark.parametrize("case", ["failing_copy", "full_device", "small_stage", "given_back"])
def test_transfers(program, case):
    r = subprocess.run([program, case], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
