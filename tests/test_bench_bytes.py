"""The byte counts of bench.py's rooflines: no more than the HBM traffic measured for
the same launches and steps (profiles/hbm_bytes_256x256x160.md), so that a roofline
fraction credits no bytes that the code does not move."""
import os
import re

import pytest

import bench
from tests.conftest import ROOT

CELLS = 256 * 256 * 160


def profile():
    with open(os.path.join(ROOT, "profiles", "hbm_bytes_256x256x160.md")) as f:
        return f.read()


@pytest.mark.parametrize("prec,elem", [("fp64", 8), ("mixed", 4)])
def test_step_bytes(prec, elem):
    section = profile().split(f"\n## {prec}\n")[1]
    measured = float(re.search(r"Per step[^:]*: ([0-9.]+) GB", section).group(1)) * 1e9
    counted = bench.step_bytes_per_cell(elem) * CELLS
    # and the halo planes and small kernels that are not counted stay a small part
    assert 0.8 * measured < counted <= measured


@pytest.mark.parametrize("kernel", ["xderiv2", "hydro"])
@pytest.mark.parametrize("prec,elem", [("fp64", 8), ("mixed", 4)])
def test_launch_bytes(kernel, prec, elem):
    assert bench.KERNEL_BYTES_PER_CELL[kernel][elem] * CELLS <= bench.measured_traffic(prec, kernel)
