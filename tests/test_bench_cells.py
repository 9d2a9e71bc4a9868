"""bench.py's figures of the cell kernel (no GPU): the bytes of a stage and of
an iteration on cell tiles, and the measured traffic of the committed counter
summary."""

import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402
from oplus2_matlab_amd import mesh as M  # noqa: E402
from oplus2_matlab_amd import op2  # noqa: E402


def test_bytes_on_cell_tiles():
    m = M.o_mesh(60, 30, "cartesian", seed=1)
    n, nodes, nb = m.ncell, m.nnode, m.nbedge
    sides = op2.KIND_BRES | op2.KIND_ADT | op2.KIND_ADT_SIDES
    # q, adt, qold read, q, adt written; x; records; boundary edges
    first = 14 * 8 * n + 16 * nodes + 16 * n + 16 * nb
    assert bench.cell_stage_bytes(m, sides, 8) == first
    assert bench.cell_stage_bytes(m, sides | op2.KIND_QOLD_IS_Q, 8) == first - 32 * n
    assert bench.cell_stage_bytes(m, sides | op2.KIND_SAVE | op2.KIND_SAVE_IN_PLACE, 8) == first
    assert bench.cell_stage_bytes(m, sides | op2.KIND_SAVE, 8) == first + 32 * n
    assert bench.iteration_bytes(m, 4) == 40 * n + 8 * nodes + 16 * n + 16 * nb


def test_traffic_of_the_cell_kernel():
    assert bench.cells_traffic(2400, 1200, 8) == pytest.approx(350.3e6)
    assert bench.cells_traffic(2400, 1200, 4) == pytest.approx(483.5e6)
    assert bench.cells_traffic(600, 300, 8) is None
    # what is measured is no less than what cannot be left out
    m = M.o_mesh(2400, 1200, "cartesian", seed=1)
    assert bench.cells_traffic(2400, 1200, 8) >= bench.iteration_bytes(m, 8)
