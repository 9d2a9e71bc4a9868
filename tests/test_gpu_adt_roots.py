"""adt_calc of the cell kernel takes its square roots and its division by cfl
without the library's scaling where the exponents allow it.  Its adt must be
that of the separate adt_calc kernel bit for bit: a quarter of a million cells
of perturbed states, side lengths of every magnitude from one end of the short
form's range to the other and beyond both (the flow does not depend on the
scale), several cfl."""

import dataclasses

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


def state(mesh, consts, dtype, q0, level):
    op2.set_graph_fusion(level)
    for loop in ("res_calc", "bres_calc"):
        op2.set_loop_config(loop, op2.STRATEGY_OWNER_GATHER, 128, 0)
    a = AF.Airfoil(mesh, consts, dtype, q0=q0, renumber=True)
    a.iterate()
    g = a.capture_iteration(2)
    a.run_graph(g, 2)
    op2.set_deferred_reductions(False)
    out = [v.copy() for v in a.fetch()]
    op2.op_exit()
    op2.op_init([], 0)
    return out


# (the sides' squared lengths are 2^(2k - 14) to 2^(2k - 5); the short form takes
# 2^-400 to 2^400 in double, 2^-50 to 2^50 in single)
@pytest.mark.parametrize("dtype,k,cfl", [
    ("double", -205, 0.9), ("double", -197, 0.9), ("double", -101, 0.7), ("double", 0, 0.9),
    ("double", 1, 1.0 / 3.0), ("double", 98, 1.1), ("double", 199, 0.9), ("double", 203, 0.9),
    ("double", 210, 0.9),
    ("float", -27, 0.9), ("float", -20, 0.9), ("float", 0, 0.9), ("float", 1, 0.7),
    ("float", 13, 1.1), ("float", 24, 0.9), ("float", 28, 0.9),
    ("float", 33, 0.9),
])
def test_adt_of_every_magnitude(runtime, dtype, k, cfl):
    print(f"[gpu] adt_calc, lengths x 2^{k}, cfl {cfl}, {dtype}", flush=True)
    mesh = M.o_mesh(720, 360, "random", seed=11)
    mesh = dataclasses.replace(mesh, x=np.ascontiguousarray(mesh.x * 2.0 ** k))
    consts = M.flow_constants().as_array().copy()
    consts[2] = cfl
    rng = np.random.Generator(np.random.PCG64(12))
    q0 = consts[6:10] * (1.0 + 0.02 * (2.0 * rng.random((mesh.ncell, 4)) - 1.0))
    s1 = state(mesh, consts, dtype, q0, op2.FUSION_STAGES)
    s0 = state(mesh, consts, dtype, q0, op2.FUSION_LOOPS)
    assert np.all(np.isfinite(s0[2])) and np.all(s0[2] > 0)
    for v1, v0 in zip(s1, s0):
        assert np.array_equal(v1, v0)
