"""A captured march that other loops cut: a loop of a user's own kernel, or an
adt_calc into a second dat, between the Runge-Kutta stages of an iteration.
The stages after the cut have not started at a save_soln, so q is not qold
there.  Every dat of a graph with stage kernels, those of the loops in between
included (they see the state at their place in the order of calls), must equal
that of a graph with res_calc and update as kernels of their own bit for bit,
on one tile, on tiles with rings and on batches."""

import ctypes
import os

import numpy as np
import pytest

from oplus2_matlab_amd import airfoil as AF
from oplus2_matlab_amd import mesh as M
from oplus2_matlab_amd import op2
from oplus2_matlab_amd.op2 import (OP_ID, OP_INC, OP_MAX, OP_MIN, OP_READ, OP_WRITE, op_arg_dat,
                                   op_arg_gbl)

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


class Between:
    """The loops called between stages, and the dats they write."""

    def __init__(self, a):
        self.a, t, n = a, a.t, a.ncell
        rng = np.random.Generator(np.random.PCG64(5))
        self.adt2 = np.zeros(n, a.real)
        self.p_adt2 = op2.op_decl_dat(a.cells, 1, t, self.adt2, "p_adt2")
        self.av = np.ascontiguousarray(rng.random((n, 3)))
        self.b = np.zeros((n, 2), np.float32)
        self.p_av = op2.op_decl_dat(a.cells, 3, "double", self.av, "p_av")
        self.p_b = op2.op_decl_dat(a.cells, 2, "float", self.b, "p_b")
        self.scale = np.array([1.5, -0.5])
        op2.op_decl_const2("gen_scale", 1, "double", np.array([2.0]))
        self.flux = np.zeros((n, 4))
        if t == "double":
            self.p_flux = op2.op_decl_dat(a.cells, 4, "double", self.flux, "p_flux")

    def adt(self):
        a, t = self.a, self.a.t
        op2.op_par_loop(None, "adt_calc", a.cells,
                        *(op_arg_dat(a.p_x, i, a.pcell, 2, t, OP_READ) for i in range(4)),
                        op_arg_dat(a.p_q, -1, OP_ID, 4, t, OP_READ),
                        op_arg_dat(self.p_adt2, -1, OP_ID, 1, t, OP_WRITE))

    def apart(self):  # a user's loop on other dats
        total, top, low = np.zeros(2, np.float32), np.array([-5], np.int32), np.array([10.0])
        op2.op_par_loop(None, "gen_direct", self.a.cells,
                        op_arg_dat(self.p_av, -1, OP_ID, 3, "double", OP_READ),
                        op_arg_dat(self.p_b, -1, OP_ID, 2, "float", OP_WRITE),
                        op_arg_gbl(self.scale, 2, "double", OP_READ),
                        op_arg_gbl(total, 2, "float", OP_INC),
                        op_arg_gbl(top, 1, "int", OP_MAX),
                        op_arg_gbl(low, 1, "double", OP_MIN))

    def reads(self):  # a user's loop that reads q and adt
        a, D = self.a, "double"
        op2.op_par_loop(None, "gen_res_calc", a.edges,
                        op_arg_dat(a.p_x, 0, a.pedge, 2, D, OP_READ),
                        op_arg_dat(a.p_x, 1, a.pedge, 2, D, OP_READ),
                        op_arg_dat(a.p_q, 0, a.pecell, 4, D, OP_READ),
                        op_arg_dat(a.p_q, 1, a.pecell, 4, D, OP_READ),
                        op_arg_dat(a.p_adt, 0, a.pecell, 1, D, OP_READ),
                        op_arg_dat(a.p_adt, 1, a.pecell, 1, D, OP_READ),
                        op_arg_dat(self.p_flux, 0, a.pecell, 4, D, OP_INC),
                        op_arg_dat(self.p_flux, 1, a.pecell, 4, D, OP_INC))

    def fetch(self):
        dats = [self.p_adt2, self.p_b] + ([self.p_flux] if self.a.t == "double" else [])
        return [op2.op_fetch_data(d).copy() for d in dats]


def march(make, level, stages, cut, at, where):
    for loop in ("res_calc", "bres_calc"):
        op2.set_loop_config(loop, op2.STRATEGY_OWNER_GATHER, 128, 0)
    op2.set_graph_fusion(level)
    a = make()
    a.iterate()
    others = Between(a)
    op2.set_deferred_reductions(True)
    getattr(others, cut)()  # (makes its plan)
    op2.reduction_log()
    op2.graph_begin()
    for _ in range(3):
        a.save_soln()
        for s in range(stages):
            if where == "update" and s == at:
                getattr(others, cut)()
            a.adt_calc()
            if where == "adt" and s == at:
                getattr(others, cut)()
            a.res_calc()
            a.bres_calc()
            a.update()
    gid = op2.graph_end()
    logs = []
    for _ in range(2):
        op2.graph_launch(gid, 2)
        logs.append(op2.reduction_log())
        a.iterate()
        op2.reduction_log()
    out = [v.copy() for v in a.fetch()] + others.fetch()
    op2.set_deferred_reductions(False)
    return np.concatenate(logs), out


def compare(make, *how):
    h1, s1 = march(make, op2.FUSION_STAGES, *how)
    op2.op_exit()
    op2.op_init([], 0)
    h0, s0 = march(make, op2.FUSION_LOOPS, *how)
    for v1, v0 in zip(s1, s0):
        assert np.array_equal(v1, v0)
    # (each rms sum adds the same positive terms in another order)
    assert h1.shape == h0.shape and np.all(np.abs(h1 - h0) <= 1e-13 * np.abs(h0))


# `at`: the stage before which the march is cut, after the update before it
# ("update") or after the stage's own adt_calc ("adt")
CUTS = [(2, 1, "update"), (2, 1, "adt"), (2, 0, "adt"), (3, 1, "update"), (3, 2, "update"),
        (4, 2, "update"), (4, 2, "adt"), (2, 0, "update")]


@pytest.mark.parametrize("dtype", ["double", "float"])
@pytest.mark.parametrize("cut", ["apart", "adt"])
@pytest.mark.parametrize("stages,at,where", CUTS)
@pytest.mark.parametrize("ni,nj", [(20, 10), (61, 37)])
def test_march_cut_in_mid_iteration(runtime, dtype, cut, stages, at, where, ni, nj):
    print(f"[gpu] march {ni}x{nj} of {stages} stages cut by {cut} at {at} after {where}, {dtype}",
          flush=True)
    mesh = M.o_mesh(ni, nj, "random", seed=6)
    compare(lambda: AF.Airfoil(mesh, M.flow_constants().as_array(), dtype, renumber=True),
            stages, cut, at, where)


@pytest.mark.parametrize("stages,at,where", CUTS)
@pytest.mark.parametrize("ni,nj", [(20, 10), (61, 37), (741, 400)])
def test_march_read_by_a_user_loop(runtime, stages, at, where, ni, nj):
    print(f"[gpu] march {ni}x{nj} of {stages} stages read at {at} after {where}", flush=True)
    mesh = M.o_mesh(ni, nj, "cartesian", seed=6)
    compare(lambda: AF.Airfoil(mesh, M.flow_constants().as_array(), "double", renumber=True),
            stages, "reads", at, where)


@pytest.mark.parametrize("dtype", ["double", "float"])
@pytest.mark.parametrize("cut", ["apart", "adt"])
def test_batch_cut_in_mid_iteration(runtime, dtype, cut):
    print(f"[gpu] batch cut by {cut}, {dtype}", flush=True)
    batch = M.mesh_batch(3, 3, 900, 4000, "random")
    compare(lambda: AF.AirfoilBatch(batch, dtype, renumber=True), 2, cut, 1, "update")
