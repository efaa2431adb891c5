"""cf_set_graph captures the pipelined sweeps and DPLUSGS only.  The other
sweep schedules, chosen by cf_set_sweep_schedule or by metrics that are not
diagonal, launch eagerly with the graph switched on: no capture is made and the
bits are those of a context without the switch."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


def _run(cfg, Q, graph, schedules, skewed=False):
    from channel_flow_amd.solver import Solver
    with Solver(cfg) as s:
        met = s.Jacobian_all(cfg.gamma_metric)
        if skewed:
            met["m"][1] += 1e-3 * met["m"][0]  # xidy of the cells: no longer diagonal
            s.set_metrics(met)
        s.set_graph(graph)
        s.load_state(Q, Q)
        ers, builds = [], []
        for schedule in schedules:
            s.set_sweep_schedule(schedule)
            ers.append(s.inner_iteration())
            builds.append(s.graph_builds())
        return np.array(ers), s.read_state()[2], builds


@pytest.mark.parametrize("schedules,skewed,builds", [((1, 2, 1, 2), False, [0, 0, 0, 0]),
                                                     ((0, 1, 2, 0, 0), False, [1, 1, 1, 1, 1]),
                                                     ((0, 2, 0), True, [0, 0, 0])])
def test_gpu_graph_leaves_other_schedules_eager(schedules, skewed, builds):
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    print(f"graph with schedules {schedules} skewed {skewed}", flush=True)
    cfg = ChannelConfig(12, 10, 16, gamma_metric=2.0, deltaT=1e-8)
    Q = poiseuille_state(cfg, FlowParams(), seed=5, stream=0)
    e0, q0, b0 = _run(cfg, Q, False, schedules, skewed)
    e1, q1, b1 = _run(cfg, Q, True, schedules, skewed)
    assert b0 == [0] * len(schedules) and b1 == builds
    np.testing.assert_array_equal(e0, e1)
    np.testing.assert_array_equal(q0, q1)
