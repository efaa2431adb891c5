"""The DPLUSGS Jacobi sweeps on grids at the edges of their blocks (64 x 4
cells, four blocks along j walking i) and on both sides of the rule that picks
the kernel: the summary of a thin grid (8x8x64) does not fit the sweep buffer's
scratch and takes the general one.  The oracle adds in the same order, so the
iterate agrees bit for bit, the norms to 1e-12."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


@pytest.mark.parametrize("grid", [(8, 8, 8), (8, 8, 64), (9, 17, 11), (10, 24, 66), (33, 9, 24)])
def test_gpu_jacobi_sweeps_match_oracle(grid):
    from oracle import oracle as O
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    from channel_flow_amd.solver import Solver
    print(f"jacobi {grid}", flush=True)
    cfg = ChannelConfig(*grid, gamma_metric=1.5, deltaT=5e-8)
    Qn = poiseuille_state(cfg, FlowParams(), seed=7, stream=0)
    Qm = poiseuille_state(cfg, FlowParams(), seed=7, stream=1)
    met = O.metrics(cfg)
    U, Uq = O.state_from_Q(cfg, Qn, met["J"]), O.state_from_Q(cfg, Qm, met["J"])
    Ui = [a.copy() for a in U]
    er_o = [O.inner_iteration(cfg, Ui, U, Uq, met, dplusgs=True) for _ in range(2)]
    sl = (slice(3, cfg.gend + 1), slice(2, cfg.ny + 1), slice(2, cfg.nz + 1))
    qi_o = np.stack([Ui[v][sl] * met["J"][sl] for v in range(5)])
    for graph in (False, True):
        with Solver(cfg) as s:
            s.set_implicit_solver(1)
            s.set_graph(graph)
            s.Jacobian_all(1.5, want_arrays=False)
            s.load_state(Qn, Qm)
            er = [s.inner_iteration() for _ in range(2)]
            qi = s.read_state()[2]
        np.testing.assert_array_equal(qi, qi_o)
        np.testing.assert_allclose(np.array(er), np.array(er_o), rtol=1e-12, atol=0)
