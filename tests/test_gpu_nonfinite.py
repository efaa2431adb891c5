"""The face fluxes and viscous terms of states that hold infinities, zero and
tiny densities or values near overflow, on host arrays: a division's results
with such operands (infinities, zeros, NaN) come back as the reference's
arithmetic gives them, cell for cell, against the oracle.  The quotients go
through reciprocals, which give NaN there, and are formed again by division.

The viscous terms are compared for infinite densities, where the velocities are
zero, in the three momentum components: the fused kernel leaves out terms with
exactly zero coefficients, which the oracle multiplies with the temperature
(NaN) in the energy's."""
import numpy as np
import pytest

from conftest import gpu_available, masks

pytestmark = pytest.mark.gpu

# field, value: rho, rho u, rho v, rho w, rho E over J
PLANTS = {"rho zero": (0, 0.0), "rho inf": (0, np.inf), "rho subnormal": (0, 1e-320), "rho 1e-308": (0, 1e-308),
          "u inf": (1, np.inf), "u 1e154": (1, 1e154), "v 1e300": (2, 1e300), "v nan": (2, np.nan),
          "E inf": (4, np.inf), "E -inf": (4, -np.inf), "E 1e305": (4, 1e305), "E 1.7e308": (4, 1.7e308)}


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


@pytest.mark.parametrize("grid", [(12, 10, 16), (21, 13, 70)])
@pytest.mark.parametrize("face_J", [1.0, 1e-8])
def test_gpu_nonfinite_faces_match_oracle(grid, face_J):
    from oracle import oracle as O
    from channel_flow_amd.config import ChannelConfig, FlowParams, poiseuille_state
    from channel_flow_amd.solver import Solver
    print(f"nonfinite {grid} face J x {face_J}", flush=True)
    cfg = ChannelConfig(*grid, gamma_metric=1.5)
    met = O.metrics(cfg)
    for q in ("J_u", "J_v", "J_w"):
        met[q] = met[q] * face_J
    U0 = O.state_from_Q(cfg, poiseuille_state(cfg, FlowParams(), seed=3, stream=0), met["J"])
    O.halo_bc(cfg, U0, met["J"])
    rng = np.random.default_rng(1)
    m = masks(cfg)
    nonfinite = 0
    with Solver(cfg) as s, np.errstate(all="ignore"):
        for name, (v, x) in PLANTS.items():
            U = [a.copy() for a in U0]
            for _ in range(3):
                U[v][rng.integers(3, cfg.gend + 1), rng.integers(2, cfg.ny + 1), rng.integers(2, cfg.nz + 1)] = x
            for d, flux in enumerate((s.Flux_X, s.Flux_Y, s.Flux_Z)):
                Jf, mf = met["J_" + "uvw"[d]], met["m_" + "uvw"[d]]
                got, want = flux(U, met["J"], Jf, mf), O.flux(cfg, d, U, met["J"], Jf, mf)
                for c in range(5):
                    a, b = got[c][m["xyz"[d]]], want[c][m["xyz"[d]]]
                    np.testing.assert_array_equal(a, b, err_msg=f"{name}: flux {d}, field {c}")
                    nonfinite += np.isinf(b).sum()
            if name == "rho inf":
                for a, b in zip(s.Viscous_terms(U, met)[:3], O.viscous(cfg, U, met)[:3]):
                    np.testing.assert_array_equal(a[m["int"]], b[m["int"]], err_msg=f"{name}: viscous terms")
    assert nonfinite > 0
