"""The stencils on four streams, which run there from 150000 cells in a graph
and from 4 million eagerly, against one after another: ragged extents, periodic
x, FP32 sweeps, DPLUSGS and the three-kernel viscous terms, on grids above those
bounds, with other work on the context's stream between the iterations."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


@pytest.mark.parametrize("periodic,precision,solver,viscous", [(False, 0, 0, 0), (True, 1, 0, 0), (True, 0, 1, 0),
                                                               (False, 0, 0, 1), (True, 0, 1, 1)])
@pytest.mark.parametrize("grid,graph", [((70, 45, 53), True), ((161, 157, 163), False)])
def test_gpu_four_streams_same_bits(grid, graph, periodic, precision, solver, viscous):
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    from channel_flow_amd.solver import Solver
    print(f"four streams {grid} graph {graph} {periodic, precision, solver, viscous}", flush=True)
    assert np.prod(grid) >= (150_000 if graph else 4_000_000)
    cfg = ChannelConfig(*grid, gamma_metric=2.0, deltaT=1e-8, x_periodic=periodic)
    Q = poiseuille_state(cfg, FlowParams(), seed=15, stream=0)
    got = []
    for concurrent in (True, False):
        with Solver(cfg, precision=precision) as s:
            s.Jacobian_all(2.0, want_arrays=False)
            s.set_implicit_solver(solver)
            s.set_viscous_schedule(viscous)
            s.set_graph(graph)
            s.set_concurrent_stencils(concurrent)
            s.load_state(Q, Q)
            er = []
            for _ in range(3):
                er.append(s.inner_iteration())
                s.Driven_force()
            assert s.graph_builds() == int(graph)
            got.append((np.array(er), s.read_state()[2]))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
