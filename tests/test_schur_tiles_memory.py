"""Host construction of the reduced camera system's structure
(maplab_amd/csrc/ba_tiles.cc): what it allocates grows with the map, not with
the square of its vertices, and the rows of S are those of a plain count."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "maplab_amd", "csrc")


def build(tmp_path_factory, name):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path_factory.mktemp("tiles") / name)
    subprocess.run([gxx, "-O2", "-std=c++17", "-pthread", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "native", name + ".cc"), os.path.join(CSRC, "ba_tiles.cc")], check=True)
    return exe


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return build(tmp_path_factory, "schur_tiles_memory")


def test_allocations_are_linear_in_the_rows(program):
    # Twice the rows with the same landmarks each: twice the bytes. A table over
    # pairs of bands (64000 rows: 128 MB) or arrays of all rows for a few rows
    # each (8 GB in all) would show in the larger system.
    small, large = ([int(x) for x in subprocess.run([program, str(n), "2"], capture_output=True, text=True,
                                                    check=True).stdout.split()] for n in (32000, 64000))
    print(small, large)
    assert large[0] < 2.2 * small[0] and large[1] < 2.2 * small[1]
    assert large[1] < 64000 * 4096


@pytest.mark.parametrize("rows, per_row", [(1, 1), (2, 5), (15, 3), (16, 3), (17, 3), (33, 1), (500, 4), (2000, 1)])
def test_rows_match_a_plain_count(program, rows, per_row):
    out = subprocess.run([program, str(rows), str(per_row), "check"], capture_output=True, text=True)
    assert out.returncode == 0, (out.returncode, out.stdout)


@pytest.mark.parametrize("rows, landmarks", [(100, 12), (100, 13), (400, 60), (700, 4500)])
def test_few_landmarks_over_many_bands(tmp_path_factory, rows, landmarks):
    # Visits sorted by tile row, then by column (fewer than a fourth as many
    # landmarks as pairs of bands, times the pieces of 4096 landmarks).
    program = build(tmp_path_factory, "schur_tiles_check")
    out = subprocess.run([program, str(rows), str(landmarks), "8"], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
