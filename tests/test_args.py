"""Loop arguments made by op2.py: type names that are not plain str, and
arrays that have no type of the runtime."""

import numpy as np
import pytest

from oplus2_matlab_amd import op2


class Name(str):
    pass


@pytest.fixture
def dat():
    op2.lib().op_init_core(0, None, 0)
    cells = op2.op_decl_set(4, "cells")
    yield op2.op_decl_dat_host(cells, 2, "double", np.zeros(8), "d")
    op2.op_exit()


@pytest.mark.parametrize("name", [str, np.str_, Name])
def test_type_name_outlives_the_call(dat, name):
    """The argument points at its type's name: whatever string gave it, the
    name is still there when the loop reads it."""
    args = [op2.op_arg_dat(dat, -1, op2.OP_ID, 2, name("double"), op2.OP_READ),
            op2.op_arg_gbl(np.zeros(1), 1, name("double"), op2.OP_READ)]
    others = [b"%06d" % i for i in range(1000)]  # (take the place of what was freed)
    assert [a.type for a in args] == [b"double"] * 2
    assert len(others) == 1000


def test_array_of_no_type(dat):
    """Refused by the loop, not by making the argument: a type the runtime
    does not have is the argument type "error" (common/op_lib.h:184-190)."""
    a = op2.op_arg_gbl(np.zeros(1, "datetime64[s]"), 1, "double", op2.OP_INC)
    assert a.type == b"error" and a.data
