"""The inner iteration's launches: the one-kernel ghost cells against the
oracle at the edges of its three thread ranges, the pre-pass's reset of the
sweep tickets over several sweep pairs, and the stencils on four streams, which
run there only on larger grids."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


@pytest.mark.parametrize("grid", [(8, 8, 8), (9, 10, 67), (13, 70, 9)])
@pytest.mark.parametrize("periodic", [False, True])
def test_gpu_ghosts_equal_the_three_passes(grid, periodic):
    """x ghost planes, then walls, then periodic z, as the reference orders
    them, restated in numpy with the walls from an x-ghost-free run."""
    from channel_flow_amd.config import ChannelConfig
    from channel_flow_amd.solver import Solver
    print(f"ghosts {grid} periodic {periodic}", flush=True)
    cfg = ChannelConfig(*grid, gamma_metric=2.0, x_periodic=periodic)
    rng = np.random.default_rng(3)
    with Solver(cfg) as s:
        J = s.Jacobian_all(2.0)["J"]
        U = [1.0 + 0.1 * rng.random(cfg.shape) for _ in range(4)] + [300.0 + rng.random(cfg.shape)]
        got = [a.copy() for a in U]
        s.boundary_conditions(got, J)
    g, ny, nz = cfg.gend, cfg.ny, cfg.nz
    lo, hi = (g, 3) if periodic else (3, g)
    want = [a.copy() for a in U]
    for w in want:
        w[2], w[g + 1] = w[lo], w[hi]
    KG, RG, TW2 = 1.4, 287.0, 2 * 298.0592
    i, k = slice(2, g + 2), slice(2, nz + 1)
    for ja, jb in ((2, 1), (ny, ny + 1)):
        U1, U2, U3, U4, U5 = (w[i, ja, k] for w in want)
        Ja, Jb = J[3, ja, 2], J[3, jb, 2]
        rho = U1 * Ja
        u, v, ww = U2 / U1, U3 / U1, U4 / U1
        VV = u * u + v * v + ww * ww
        P = (U5 * Ja - 0.5 * rho * VV) * (KG - 1)
        T = TW2 - P / rho / RG
        rho = P / RG / T
        new = (P / RG / T / Jb, -P / RG / T * u / Jb, -P / RG / T * v / Jb, -P / RG / T * ww / Jb,
               (rho * RG * T / (KG - 1) + 0.5 * P / RG / T * VV) / Jb)
        for w, n in zip(want, new):
            w[i, jb, k] = n
    for w in want:
        w[i, :ny + 3, 1] = w[i, :ny + 3, nz]
        w[i, :ny + 3, nz + 1] = w[i, :ny + 3, 2]
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("grid,graph", [((64, 48, 56), True), ((192, 144, 160), False)])
def test_gpu_stencils_on_four_streams_same_bits(grid, graph):
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    from channel_flow_amd.solver import Solver
    print(f"four streams {grid} graph {graph}", flush=True)
    cfg = ChannelConfig(*grid, gamma_metric=2.0, deltaT=1e-8, n_sweeps=3)
    Q = poiseuille_state(cfg, FlowParams(), seed=10, stream=0)
    runs = []
    for concurrent in (True, False):
        with Solver(cfg) as s:
            s.Jacobian_all(2.0, want_arrays=False)
            s.set_graph(graph)
            s.set_concurrent_stencils(concurrent)
            s.set_sweep_reuse(concurrent)  # three sweep pairs in the other run
            s.load_state(Q, Q)
            runs.append((np.array([s.inner_iteration() for _ in range(2)]), s.read_state()[2]))
    np.testing.assert_array_equal(runs[0][0], runs[1][0])
    np.testing.assert_array_equal(runs[0][1], runs[1][1])
