"""The splitting of admission's host work over threads (in_pieces), where memory
runs out or a piece throws: checked on the host in a small program."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "simbody_amd")


def test_every_piece_is_done(tmp_path):
    if not os.path.exists(os.path.join(LIB, "libtdyn.so")):
        pytest.skip("library not built")
    hip = os.environ.get("ROCM_PATH", "/opt/rocm")
    if shutil.which("g++") is None or not os.path.isdir(os.path.join(hip, "include", "hip")):
        pytest.skip("no host compiler or HIP headers")
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(hip, "include"),
                    os.path.join(HERE, "in_pieces_check.cpp"), "-o", exe, "-L", LIB, "-ltdyn", "-Wl,-rpath," + LIB,
                    "-L", os.path.join(hip, "lib"), "-lamdhip64", "-Wl,-rpath," + os.path.join(hip, "lib"), "-lpthread"],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
