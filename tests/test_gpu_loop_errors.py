"""op_par_loop reports what the runtime records while a loop runs: the argument
checks at OP_diags >= 1 (common/op_lib_core.c:266-305), which do not keep the
loop from running."""

import ctypes
import os

import numpy as np
import pytest

from oplus2_matlab_amd import op2
from oplus2_matlab_amd.op2 import (OP_ID, OP_INC, OP_MAX, OP_MIN, OP_READ, OP_WRITE, op_arg_dat,
                                   op_arg_gbl)

pytestmark = pytest.mark.gpu


@pytest.fixture
def cells():
    ctypes.CDLL(os.path.join(os.path.dirname(op2.LIB_PATH), "libop2_testloops.so"),
                mode=ctypes.RTLD_GLOBAL)
    op2.op_init([], 1)
    yield op2.op_decl_set(300, "cells")
    op2.op_exit()


def test_type_other_than_the_dat(cells):
    print("[gpu] save_soln with arguments of another type, OP_diags 1", flush=True)
    q = op2.op_decl_dat(cells, 4, "double", np.ones((300, 4)), "q")
    qold = op2.op_decl_dat(cells, 4, "double", np.zeros((300, 4)), "qold")

    def loop(typ):
        op2.op_par_loop(None, "save_soln", cells,
                        op_arg_dat(q, -1, OP_ID, 4, typ, OP_READ),
                        op_arg_dat(qold, -1, OP_ID, 4, typ, OP_WRITE))

    loop("double")
    with pytest.raises(op2.OP2Error, match="type does not match"):
        loop("float")
    loop("double")  # (an error reported is an error forgotten)
    assert np.array_equal(op2.op_fetch_data(qold), np.ones((300, 4)))


def test_dim_other_than_the_dat(cells):
    print("[gpu] a user's loop with an argument of another dim, OP_diags 1", flush=True)
    op2.op_decl_const2("gen_scale", 1, "double", np.array([2.0]))
    a = op2.op_decl_dat(cells, 3, "double", np.ones((300, 3)), "a")
    b = op2.op_decl_dat(cells, 2, "float", np.zeros((300, 2), np.float32), "b")
    scale = np.array([1.5, -0.5])

    def loop(dim):
        total, top, low = np.zeros(2, np.float32), np.array([-5], np.int32), np.array([10.0])
        op2.op_par_loop(None, "gen_direct", cells,
                        op_arg_dat(a, -1, OP_ID, dim, "double", OP_READ),
                        op_arg_dat(b, -1, OP_ID, 2, "float", OP_WRITE),
                        op_arg_gbl(scale, 2, "double", OP_READ),
                        op_arg_gbl(total, 2, "float", OP_INC),
                        op_arg_gbl(top, 1, "int", OP_MAX),
                        op_arg_gbl(low, 1, "double", OP_MIN))

    loop(3)
    with pytest.raises(op2.OP2Error, match="dim does not match"):
        loop(2)
    loop(3)
    assert np.array_equal(op2.op_fetch_data(b), np.tile(np.float32([2.5, -1.0]), (300, 1)))
