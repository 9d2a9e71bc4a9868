"""A loop with increments and a direct result whose targets take too many
elements for a tile is left to the coloured plan.  That is asked at every call
of the loop; the map is looked through at the first alone."""

import time

import numpy as np
import pytest

from oplus2_matlab_amd import op2
from oplus2_matlab_amd.op2 import OP_ID, OP_INC, OP_WRITE, op_arg_dat

N = 4_000_000


@pytest.fixture
def program():
    op2.lib().op_init_core(0, None, 0)
    yield
    op2.op_exit()


def keeps(ntarget, part=0, n=N, name="edge_loop"):
    """The call for n edges to ntarget zones, as the generic path makes it."""
    edges, zones = op2.op_decl_set(n, "edges"), op2.op_decl_set(ntarget, "zones")
    m = op2.op_decl_map(edges, zones, 1, np.arange(n, dtype=np.int32) % ntarget, "zone")
    total = op2.op_decl_dat_host(zones, 1, "double", np.zeros(ntarget), "total")
    out = op2.op_decl_dat_host(edges, 1, "float", np.zeros(n, np.float32), "out")
    args = (op2.OpArg * 2)(op_arg_dat(total, 0, m, 1, "double", OP_INC),
                           op_arg_dat(out, -1, OP_ID, 1, "float", OP_WRITE))

    def call():
        """Whether the loop is refused (no plan, no error), and the seconds that took."""
        op2.lib().op2_clear_error()
        t = time.perf_counter()
        got = op2.lib().op2_generic_owner_keeps(name.encode(), edges._p, 2, args, part)
        return not got and not op2.lib().op2_last_error(), time.perf_counter() - t

    return call


def test_refusal_is_remembered(program):
    call = keeps(500)
    refused, first = call()
    assert refused
    again = [call() for _ in range(5)]
    assert all(r for r, _ in again)
    # (a pass over the map is about 5 ms; without one, a call takes a few us)
    assert min(t for _, t in again) < first / 20


def test_bound_of_each_map_and_part(program):
    """At most 16383 elements a tile: the answer is a map's and a part size's
    own, and the next program's maps are its own.  (Without a GPU a loop that
    is not refused fails to upload its plan.)"""
    n = 50_000
    assert keeps(300, n=n)()[0]                # 167 elements a target, 128 targets
    small = keeps(1000, n=n, name="other")     # 50
    assert not small()[0] and not small()[0]
    assert keeps(1000, part=512, n=n, name="third")()[0]
    op2.op_exit()
    op2.lib().op_init_core(0, None, 0)
    assert not keeps(1000, n=n, name="other")()[0]
    assert keeps(300, n=n)()[0]
