"""The host side of the downloads (csrc/isph_transfer.hip) on the CPU: built as
the library is and linked with a stand-in for the HIP runtime
(transfer_host.cpp), so that contexts, streams and devices can be arranged that
one GPU does not have."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "beach_slope_confined_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    sys.path.insert(0, os.path.dirname(HERE))
    from __graft_entry__ import HIP_FLAGS
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    out = tmp_path_factory.mktemp("transfer")
    for src, obj, flags in ((os.path.join(CSRC, "isph_transfer.hip"), "transfer.o", []),
                            (os.path.join(HERE, "transfer_host.cpp"), "host.o",
                             ["-x", "hip", "--offload-host-only"])):
        subprocess.run([hipcc] + HIP_FLAGS + flags + ["-I", CSRC, "-c", src, "-o",
                                                      str(out / obj)], check=True)
    exe = str(out / "transfer_host")
    subprocess.run(["g++", str(out / "transfer.o"), str(out / "host.o"), "-o", exe, "-pthread"],
                   check=True)
    return exe


@pytest.mark.parametrize("scenario", ["busy", "busy_unpinned", "crowd", "device"])
def test_downloads(program, scenario):
    r = subprocess.run([program, scenario], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
