"""Which stages of a capture are timed (op2_set_graph_kernel_timing): those
numbered n, 2n, ..., each with the loops that its kernel runs, whatever the
number of stages in an iteration and of iterations in a launch."""

import pytest

from oplus2_matlab_amd import airfoil as AF
from oplus2_matlab_amd import mesh as M
from oplus2_matlab_amd import op2

pytestmark = pytest.mark.gpu

ITERATIONS = 5


@pytest.fixture
def runtime():
    op2.op_init([], 0)
    for loop in ("res_calc", "bres_calc"):
        op2.set_loop_config(loop, op2.STRATEGY_OWNER_GATHER, 128, 0)
    yield
    op2.set_graph_kernel_timing(0)
    op2.set_deferred_reductions(False)
    op2.op_exit()
    op2.set_loop_config(None, 0, 0, 0)


@pytest.mark.parametrize("stages", [1, 2, 3])
@pytest.mark.parametrize("every", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("ni,nj", [(20, 10), (61, 37)])
def test_timed_stages(runtime, stages, every, ni, nj):
    print(f"[gpu] {ni}x{nj}, {stages} stages an iteration, every {every}th timed", flush=True)
    a = AF.Airfoil(M.o_mesh(ni, nj, "random", seed=6), M.flow_constants().as_array(), "double",
                   renumber=True)
    a.iterate()
    op2.set_deferred_reductions(True)
    op2.set_graph_kernel_timing(every)
    op2.graph_begin()
    for _ in range(ITERATIONS):
        a.save_soln()
        for _ in range(stages):
            a.adt_calc()
            a.res_calc()
            a.bres_calc()
            a.update()
    gid = op2.graph_end()
    op2.graph_launch(gid, 2)
    got = op2.graph_kernel_times(gid)
    total = ITERATIONS * stages
    timed = range(every, total + 1, every)
    # 1 bres_calc, 2 the next iteration's save_soln, 4 the adt_calc that follows
    want = [1 + 2 * (n % stages == 0 and n < total) + 4 * (n < total) for n in timed]
    assert [k & 7 for k, _ in got] == want
    assert all(ms > 0 for _, ms in got)
