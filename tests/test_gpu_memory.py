"""Device memory of a context, which bounds the grids that fit: 52 fields of
the padded layout and 24 in sweep order (tiles of 8 x 8 columns, Z + 14 steps
of 64 lanes).  The sweeps' hand-off slots and edge copies share memory with the
fields that the same schedule does not use, so the schedules are also switched
between sweep pairs that do use it."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


@pytest.mark.parametrize("precision", [0, 1])
def test_gpu_context_memory(precision):
    import torch
    from channel_flow_amd.config import ChannelConfig
    from channel_flow_amd.solver import Solver
    print(f"context memory, precision {precision}", flush=True)
    Solver(ChannelConfig(16, 12, 16), precision=precision).close()
    X, Y, Z = 128, 96, 128
    cfg = ChannelConfig(X, Y, Z)
    before = torch.cuda.mem_get_info()[0]
    with Solver(cfg, precision=precision):
        used = before - torch.cuda.mem_get_info()[0]
    Xnp, Ym, Zm = cfg.shape
    field = Xnp * Ym * (-(-Zm // 8) * 8)
    sweep = -(-X // 8) * -(-Y // 8) * (Z + 14) * 64
    # 20 MB for profiles, partials and the allocator's rounding (one more
    # field in sweep order is 14 MB)
    assert used <= 8 * (52 * field + 24 * sweep) + 20e6, (used, 8 * field, 8 * sweep)


@pytest.mark.parametrize("grid", [(8, 8, 8), (17, 25, 11)])
def test_gpu_sweep_pairs_and_schedules_share_memory(grid):
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    from channel_flow_amd.solver import Solver
    print(f"pairs and schedules {grid}", flush=True)
    cfg = ChannelConfig(*grid, gamma_metric=2.0, deltaT=1e-8, n_sweeps=3)
    Q = poiseuille_state(cfg, FlowParams(), seed=13, stream=0)
    got = []
    for order, reuse in (((1, 1, 1, 1, 1, 1), True), ((0, 2, 0, 2, 2, 0), False)):
        with Solver(cfg) as s:
            s.Jacobian_all(cfg.gamma_metric, want_arrays=False)
            s.set_sweep_reuse(reuse)
            s.load_state(Q, Q)
            for schedule in order:
                s.set_sweep_schedule(schedule)
                s.inner_iteration()
                s.Jacobian_all(cfg.gamma_metric)
            got.append(s.read_state()[2])
    np.testing.assert_array_equal(got[0], got[1])
