"""Host arrays that pass through the staging copy in more than one piece: a
thin FP32 context (8x8x64) stages three of five fields at a time.  A null array
is named by its place in the caller's list, and every field arrives."""
import ctypes

import numpy as np
import pytest

from conftest import gpu_available

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


def _state(cfg):
    rng = np.random.default_rng(4)
    return [1.0 + 0.1 * rng.random(cfg.shape) for _ in range(4)] + [300.0 + rng.random(cfg.shape)]


@pytest.mark.parametrize("null", [0, 2, 3, 4])
@pytest.mark.parametrize("precision", [0, 1])
def test_gpu_null_array_is_named_by_its_place(null, precision):
    from channel_flow_amd.config import ChannelConfig
    from channel_flow_amd.solver import Solver
    print(f"null array {null} precision {precision}", flush=True)
    cfg = ChannelConfig(8, 8, 64)
    P = ctypes.POINTER(ctypes.c_double)
    with Solver(cfg, precision=precision) as s:
        J = s.Jacobian_all(2.0)["J"]
        U = _state(cfg)
        ptr = (P * 5)(*[None if v == null else a.ctypes.data_as(P) for v, a in enumerate(U)])
        assert s.lib.cf_boundary_conditions(s._h, ptr, J.ctypes.data_as(P)) != 0
        assert s.lib.cf_last_error(s._h).decode().endswith(f"null input array {null}")


def test_gpu_fields_in_pieces_arrive_whole():
    from channel_flow_amd.config import ChannelConfig
    from channel_flow_amd.solver import Solver
    print("fields in pieces", flush=True)
    got = []
    for precision in (0, 1):
        cfg = ChannelConfig(8, 8, 64)
        with Solver(cfg, precision=precision) as s:
            J = s.Jacobian_all(2.0)["J"]
            U = _state(cfg)
            s.boundary_conditions(U, J)
            got.append(U)
    np.testing.assert_array_equal(got[0], got[1])
