"""Work lists longer than one launch: the launchers of device.hip, compiled for the host and linked with
a stand-in for the HIP runtime, cut them into launches that the device accepts and that cover them."""
import os
import subprocess

import pytest

from qcmaquis_amd import build
from tests import emu


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="hipcc is not installed")
def test_launch_pieces(tmp_path):
    objs = []
    for src in (os.path.join(build.CSRC, "device.hip"), os.path.join(emu.HERE, "launch_pieces.cpp")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run([build.HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-I", os.path.join(build.ROOT, "include"),
                        "-I", build.CSRC, "-x", "hip", "-c", src, "-o", objs[-1]], check=True)
    prog = str(tmp_path / "launch_pieces")
    # the device code of the host-only object is nowhere: its symbol stays unresolved
    subprocess.run(["g++", "-no-pie", "-o", prog] + objs + ["-Wl,--unresolved-symbols=ignore-all"], check=True)
    r = subprocess.run([prog], capture_output=True, text=True, timeout=60)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and "gemm items" in r.stdout
