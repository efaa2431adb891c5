"""cf_profile_inner_iteration runs the LU-SGS sweeps whatever implicit solver
is set.  On a context that has never swept, its hand-off slots must be seeded
all the same: the state and norms are those of a context with the LU-SGS
solver."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


@pytest.mark.parametrize("precision", [0, 1])
def test_gpu_profile_seeds_the_sweeps_for_either_solver(precision):
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    from channel_flow_amd.solver import Solver
    print(f"profile with either solver, precision {precision}", flush=True)
    cfg = ChannelConfig(40, 33, 18, gamma_metric=2.0, deltaT=1e-8)
    Q = poiseuille_state(cfg, FlowParams(), seed=14, stream=0)
    got = []
    for solver in (0, 1):
        with Solver(cfg, precision=precision) as s:
            s.Jacobian_all(2.0, want_arrays=False)
            s.set_implicit_solver(solver)
            s.load_state(Q, Q)
            er = [s.profile_inner_iteration()[0] for _ in range(2)]
            got.append((np.array(er), s.read_state()[2]))
    np.testing.assert_array_equal(got[0][0], got[1][0])
    np.testing.assert_array_equal(got[0][1], got[1][1])
