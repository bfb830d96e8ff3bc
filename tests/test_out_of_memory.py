"""The C entry points where memory runs out: a status, never an exception
through the C interface."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "maplab_amd")


def test_create_and_masks_return_a_status(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path / "out_of_memory")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    "-I", os.path.join(os.path.dirname(HERE), "include"), "-o", exe,
                    os.path.join(HERE, "native", "out_of_memory.cc"), "-L", PKG, "-lmaplab_ba",
                    "-Wl,-rpath," + PKG, "-Wl,--allow-shlib-undefined", "-rdynamic"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(out.stdout)
    assert out.returncode == 0, (out.returncode, out.stdout, out.stderr)
