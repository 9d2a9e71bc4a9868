"""Batched updates whose cell -> mesh map is the program's own: parts of one
connected mesh.  The tiles of large FP64 meshes take two plan blocks each, and
a part that starts at the second of the two must not have its cells counted for
the part before.  Each part's rms against the sums of res_calc and update as
kernels of their own, for parts that start at an even block, at an odd one and
inside a block."""

import numpy as np
import pytest

from oplus2_matlab_amd import airfoil as AF
from oplus2_matlab_amd import mesh as M
from oplus2_matlab_amd import op2

pytestmark = pytest.mark.gpu


@pytest.fixture
def runtime():
    op2.op_init([], 0)
    yield
    op2.set_graph_fusion(True)
    op2.set_deferred_reductions(False)
    op2.op_exit()
    op2.set_loop_config(None, 0, 0, 0)


def labelled(mesh, starts):
    """The mesh as a batch: part i is the cells from starts[i] of the
    runtime's own numbering."""
    a = AF.Airfoil(mesh, M.flow_constants().as_array(), "double", renumber=True)
    at = op2.renumber_export(a.cells)
    op2.op_exit()
    op2.op_init([], 0)
    cmesh = (np.searchsorted(starts, at, side="right") - 1).astype(np.int32)
    consts = M.flow_constants().as_array()
    return M.MeshBatch(union=mesh, meshes=[mesh] * len(starts), consts=[consts] * len(starts),
                       cmesh=cmesh, bmesh=np.ascontiguousarray(cmesh[mesh.becell.reshape(-1)]),
                       qinf=np.tile(consts[6:10], (len(starts), 1)),
                       cell_off=np.concatenate([[0], np.cumsum(np.bincount(cmesh))]))


def march(batch, level):
    for loop in ("res_calc", "bres_calc"):
        op2.set_loop_config(loop, op2.STRATEGY_OWNER_GATHER, 128, 0)
    op2.set_graph_fusion(level)
    a = AF.AirfoilBatch(batch, "double", renumber=True)
    a.iterate()
    g = a.capture_iteration(2)
    hist = a.run_graph(g, 4)
    op2.set_deferred_reductions(False)
    out = [v.copy() for v in a.fetch()]
    op2.op_exit()
    op2.op_init([], 0)
    return hist, out


@pytest.mark.parametrize("ni,nj", [(741, 400), (120, 60)])
@pytest.mark.parametrize("starts", [[0, 512], [0, 256], [0, 256 * 9, 256 * 20, 256 * 23],
                                    [0, 256 * 8, 256 * 8 + 100]])
def test_parts_of_one_mesh(runtime, ni, nj, starts):
    print(f"[gpu] parts of a {ni}x{nj} mesh from {starts}", flush=True)
    batch = labelled(M.o_mesh(ni, nj, "cartesian", seed=6), starts)
    h1, s1 = march(batch, op2.FUSION_STAGES)
    h0, s0 = march(batch, op2.FUSION_LOOPS)
    for v1, v0 in zip(s1, s0):
        assert np.array_equal(v1, v0)
    # (each sum adds the same positive terms in another order)
    assert np.all(np.abs(h1 - h0) <= 1e-13 * np.abs(h0))
