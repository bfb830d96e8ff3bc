"""The reduced camera system's work decomposition does not depend on the number
of threads that build it (maplab_amd/csrc/ba_tiles.cc)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "maplab_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path_factory.mktemp("tiles") / "schur_tiles_threads")
    subprocess.run([gxx, "-O2", "-std=c++17", "-pthread", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "native", "schur_tiles_threads.cc"), os.path.join(CSRC, "ba_tiles.cc")],
                   check=True)
    return exe


@pytest.mark.parametrize("pvar, landmarks", [(1, 0), (1, 50), (16, 1), (17, 3000), (300, 60000), (40, 40000)])
def test_decomposition_is_the_same_on_one_cpu(program, pvar, landmarks):
    out = subprocess.run([program, str(pvar), str(landmarks), "3"], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
