"""The HBM traffic that bench.py reports beside its kernels comes from a
committed counter summary; it has to be of the present kernels."""
import os
import re

import pytest

import bench

HERE = os.path.dirname(os.path.abspath(__file__))
DEFAULT = {"k_schur_blocks", "k_pcg_step", "k_schur_factors", "k_linearize", "k_back_substitute"}
OBSERVATIONS, LANDMARKS = 2082331, 200000  # of the default workload


def summary():
    rows = {}
    for line in open(bench.TRAFFIC_PROFILE):
        cells = [c.strip().strip("`") for c in line.strip().strip("|").split("|")]
        if len(cells) == 7 and cells[0].startswith("mlba::"):
            rows[cells[0]] = float(cells[5])
    return rows


@pytest.mark.parametrize("kernel", sorted(DEFAULT))
def test_every_kernel_of_the_default_workload_has_traffic(kernel):
    assert bench.TRAFFIC_KERNEL[kernel] in summary()
    assert bench.measured_traffic(kernel) > 0


def test_summary_has_the_present_record():
    # The byte model of the kernels that write and read the observation records.
    header = open(os.path.join(os.path.dirname(HERE), "maplab_amd", "csrc", "ba_device.h")).read()
    record = 8 * int(re.search(r"constexpr int kObsRecord = (\d+);", header).group(1))
    rows = summary()
    assert rows["mlba::k_linearize<true, false>"] == pytest.approx(
        (OBSERVATIONS * (36 + record) + LANDMARKS * 176) / 1e6, abs=0.01)
    assert rows["mlba::k_back_substitute<false>"] == pytest.approx(
        (OBSERVATIONS * record + LANDMARKS * 216) / 1e6, abs=0.01)
