"""The pipelined sweeps' hand-off slots across everything that can leave them
in another state: grids of one tile, of lone last columns, of single rows of
tiles, and switches between the sweep schedules on one context (the
single-wave tiles hand over through NL itself, which the pipelined sweeps
fill).  Every schedule gives the same bits, so any order of schedules must."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


@pytest.mark.parametrize("grid", [(8, 8, 8), (9, 17, 11), (24, 8, 9), (8, 25, 31)])
def test_gpu_schedule_switches_keep_the_bits(grid):
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    from channel_flow_amd.solver import Solver
    print(f"schedule switches {grid}", flush=True)
    cfg = ChannelConfig(*grid, gamma_metric=2.0, deltaT=1e-8)
    Q = poiseuille_state(cfg, FlowParams(), seed=12, stream=0)
    states = []
    for order in ((1, 1, 1, 1, 1, 1, 1), (0, 2, 0, 1, 2, 2, 0)):
        with Solver(cfg) as s:
            s.Jacobian_all(cfg.gamma_metric, want_arrays=False)
            s.load_state(Q, Q)
            for schedule in order:
                s.set_sweep_schedule(schedule)
                s.inner_iteration()
            states.append(s.read_state()[2])
    np.testing.assert_array_equal(states[0], states[1])


@pytest.mark.parametrize("precision", [0, 1])
def test_gpu_host_arrays_between_iterations_leave_the_sweeps_alone(precision):
    """The staging of host arrays shares memory with the sweeps' fields, which
    take half of it in FP32: arrays that pass through it between two
    iterations change nothing."""
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    from channel_flow_amd.solver import Solver
    print(f"host arrays between iterations, precision {precision}", flush=True)
    cfg = ChannelConfig(40, 36, 24, gamma_metric=2.0, deltaT=1e-8)
    Q = poiseuille_state(cfg, FlowParams(), seed=11, stream=0)
    got = []
    for between in (False, True):
        with Solver(cfg, precision=precision) as s:
            s.Jacobian_all(2.0, want_arrays=False)
            s.load_state(Q, Q)
            er = []
            for _ in range(3):
                er.append(s.inner_iteration())
                if between:
                    s.Jacobian_all(2.0)
                    s.read_state()
            got.append((np.array(er), s.read_state()[2]))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
