"""Constants declared again during a capture (a ramp of cfl over the
iterations, of eps over the stages): every loop runs with the values that held
when it was called, also where the capture launches it later, with others or
as part of a march.  Bit for bit as kernels of their own, which on these
meshes (no cell with two boundary edges) compute what the loops fused in pairs
do."""

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


def march(make, level, ramp, at):
    """Four iterations in a capture, `ramp` times 2, 3, ... of the declared
    value from place `at` of each stage on; two replays."""
    for loop in ("res_calc", "bres_calc"):
        op2.set_loop_config(loop, op2.STRATEGY_OWNER_GATHER, 128, 0)
    op2.set_graph_fusion(level)
    a = make()
    a.iterate()
    base = dict(zip(("gam", "gm1", "cfl", "eps"), M.flow_constants().as_array()))[ramp]
    step = [0]

    def change(place, s):
        if place != at or (ramp == "cfl" and s):  # (cfl: once an iteration)
            return
        step[0] += 1
        op2.op_decl_const2(ramp, 1, a.t, np.array([base * (1.0 + 0.01 * step[0])], a.real))

    op2.set_deferred_reductions(True)
    op2.graph_begin()
    for _ in range(4):
        change("save", 0)
        a.save_soln()
        for s in range(2):
            change("adt", s)
            a.adt_calc()
            change("res", s)
            a.res_calc()
            change("bres", s)
            a.bres_calc()
            change("update", s)
            a.update()
    gid = op2.graph_end()
    op2.op_decl_const2(ramp, 1, a.t, np.array([base], a.real))
    op2.reduction_log()
    op2.graph_launch(gid, 2)
    log = op2.reduction_log()
    op2.set_deferred_reductions(False)
    return log, [v.copy() for v in a.fetch()]


@pytest.mark.parametrize("dtype", ["double", "float"])
@pytest.mark.parametrize("ramp", ["cfl", "eps", "gm1"])
@pytest.mark.parametrize("at", ["save", "adt", "res", "bres", "update"])
@pytest.mark.parametrize("ni,nj", [(20, 10), (61, 37)])
def test_constants_of_the_call(runtime, dtype, ramp, at, ni, nj):
    if ramp != "cfl" and "libop2_testloops" in open("/proc/self/maps").read():
        # (OP2_DEVICE_CONST in tests/generic_loops.hip: the copy waits for the stream)
        pytest.skip("a constant with a device copy is refused during a capture")
    print(f"[gpu] capture {ni}x{nj}, {ramp} changed before {at}, {dtype}", flush=True)
    mesh = M.o_mesh(ni, nj, "random", seed=6)

    def run(level):
        got = march(lambda: AF.Airfoil(mesh, M.flow_constants().as_array(), dtype,
                                       renumber=True), level, ramp, at)
        op2.op_exit()
        op2.op_init([], 0)
        return got

    h0, s0 = run(False)
    for level in (op2.FUSION_LOOPS, op2.FUSION_STAGES):
        h1, s1 = run(level)
        for v1, v0 in zip(s1, s0):
            assert np.array_equal(v1, v0)
        # (each sum adds the same positive terms in another order)
        assert np.all(np.abs(h1 - h0) <= 1e-13 * np.abs(h0))


def test_same_constants_cut_nothing(runtime):
    """A constant declared again with its value leaves the march whole: the
    stages' numbers of the timed kernels are as without."""
    print("[gpu] capture 61x37, constants declared again unchanged", flush=True)
    mesh = M.o_mesh(61, 37, "random", seed=6)
    consts = M.flow_constants().as_array()
    got = []
    for again in (False, True):
        a = AF.Airfoil(mesh, consts, "double", renumber=True)
        a.iterate()
        op2.set_deferred_reductions(True)
        op2.set_graph_kernel_timing(3)
        op2.graph_begin()
        for _ in range(3):
            if again:
                op2.op_decl_const2("cfl", 1, "double", consts[2:3])
            a.save_soln()
            for _ in range(2):
                a.adt_calc()
                a.res_calc()
                a.bres_calc()
                a.update()
        gid = op2.graph_end()
        op2.set_graph_kernel_timing(0)
        op2.graph_launch(gid, 2)
        got.append([k for k, _ in op2.graph_kernel_times(gid)])
        op2.set_deferred_reductions(False)
        op2.op_exit()
        op2.op_init([], 0)
    assert got[0] == got[1] and len(got[0]) == 2
