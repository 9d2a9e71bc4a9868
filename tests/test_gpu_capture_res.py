"""Captures whose res other code may write (the program has taken its device
pointer, or a user's own loop has added to it): res_calc reads it then, so the
update before must have stored its zeros.  Every fusion level bit for bit as
kernels of their own."""

import ctypes
import os

import numpy as np
import pytest

from oplus2_matlab_amd import airfoil as AF
from oplus2_matlab_amd import mesh as M
from oplus2_matlab_amd import op2
from oplus2_matlab_amd.op2 import OP_INC, OP_READ, op_arg_dat

pytestmark = pytest.mark.gpu


@pytest.fixture
def runtime():
    op2.op_init([], 0)
    ctypes.CDLL(os.path.join(os.path.dirname(op2.LIB_PATH), "libop2_testloops.so"),
                mode=ctypes.RTLD_GLOBAL)
    yield
    op2.set_graph_fusion(True)
    op2.set_deferred_reductions(False)
    op2.op_exit()
    op2.set_loop_config(None, 0, 0, 0)


def source(a):
    """A user's loop that adds to res."""
    D = "double"
    op2.op_par_loop(None, "gen_res_calc", a.edges,
                    op_arg_dat(a.p_x, 0, a.pedge, 2, D, OP_READ),
                    op_arg_dat(a.p_x, 1, a.pedge, 2, D, OP_READ),
                    op_arg_dat(a.p_q, 0, a.pecell, 4, D, OP_READ),
                    op_arg_dat(a.p_q, 1, a.pecell, 4, D, OP_READ),
                    op_arg_dat(a.p_adt, 0, a.pecell, 1, D, OP_READ),
                    op_arg_dat(a.p_adt, 1, a.pecell, 1, D, OP_READ),
                    op_arg_dat(a.p_res, 0, a.pecell, 4, D, OP_INC),
                    op_arg_dat(a.p_res, 1, a.pecell, 4, D, OP_INC))


def march(mesh, dtype, level, form):
    for loop in ("res_calc", "bres_calc"):
        op2.set_loop_config(loop, op2.STRATEGY_OWNER_GATHER, 128, 0)
    op2.set_graph_fusion(level)
    a = AF.Airfoil(mesh, M.flow_constants().as_array(), dtype, renumber=True)
    a.iterate()
    op2.set_deferred_reductions(True)
    if form == "pointer":
        a.p_res.device_ptr()
    else:
        source(a)
        a.update()
    op2.reduction_log()
    op2.graph_begin()
    for it in range(3):
        a.save_soln()
        for s in range(2):
            a.adt_calc()
            if form == "loop" and it != 1 and s == 0:
                source(a)
            a.res_calc()
            a.bres_calc()
            a.update()
    gid = op2.graph_end()
    op2.graph_launch(gid, 2)
    log = op2.reduction_log()
    op2.set_deferred_reductions(False)
    out = [v.copy() for v in a.fetch()]
    op2.op_exit()
    op2.op_init([], 0)
    return log, out


@pytest.mark.parametrize("dtype,form", [("double", "pointer"), ("float", "pointer"),
                                        ("double", "loop")])
@pytest.mark.parametrize("ni,nj", [(20, 10), (61, 37)])
def test_res_that_other_code_writes(runtime, dtype, form, ni, nj):
    print(f"[gpu] capture {ni}x{nj}, res written by others ({form}), {dtype}", flush=True)
    mesh = M.o_mesh(ni, nj, "random", seed=6)
    h0, s0 = march(mesh, dtype, False, form)
    for level in (op2.FUSION_LOOPS, op2.FUSION_STAGES):
        h1, s1 = march(mesh, dtype, level, form)
        for v1, v0 in zip(s1, s0):
            assert np.array_equal(v1, v0)
        # (each sum adds the same positive terms in another order)
        assert np.all(np.abs(h1 - h0) <= 1e-13 * np.abs(h0))
