"""The workloads this framework's speed is measured on.

Each case is one thing a user's program does through the public entry points:
physical steps of the dual-time solver on the device-resident state (the small
grid of a smoke run up to the 256x192x256 benchmark grid, FP64 and FP32 sweeps,
eager and as a replayed graph, every initial iterate), the explicit RK3 and the
DPLUSGS variants, the per-function entry points that a reference driver calls
with host arrays, and the training of the learned initial iterate.

`listed()` names the fixed cases, `draw(rng)` gives further ones of the same
ranges, `prepare` builds what the program holds before the call, `run` is one
pass, `work` the bytes and operations a pass cannot do without and `exact` the
64-bit value of the outputs where plain torch gives one.
"""
import ctypes
import math
from pathlib import Path

import numpy as np
import torch

import channel_flow_amd
from channel_flow_amd.config import FlowParams, cell_y
from channel_flow_amd.learned import channel_cfg, load
from channel_flow_amd.solver import CF_FP32_SWEEPS, CF_FP64, CF_PRED_NPARAM, Predictor, Solver

WEIGHTS = Path(channel_flow_amd.__file__).resolve().parent / "weights"
GAS, R_GAS, T_WALL = 1.4, 287.0, 298.0592


def listed():
    return [
        # a smoke run: the smallest grid of the tests, the three inner
        # iterations a physical step takes under the reference's loose test;
        # launches and the host's turnaround count
        step("smoke_16", 16, 12, 16, its=3),
        # an ordinary small channel: 20 inner iterations a step, launched eagerly
        step("step_64", 64, 64, 64, its=20, dt=5e-8),
        # odd extents (partial tiles everywhere), true periodic x
        step("ragged_periodic", 97, 75, 130, its=12, periodic=True),
        # the benchmark grid, all FP64, replayed as a graph
        step("bench_fp64", 256, 192, 256, its=60, graph=True),
        # the benchmark grid with FP32 sweeps from the cubic extrapolation:
        # the fast path of a production run past its transient
        step("bench_fp32_cubic", 256, 192, 256, its=60, graph=True, fp32=True, guess=2, order=3),
        # steps started by the network (inference, its check, the fallback)
        step("learned_64", 64, 64, 64, its=8, dt=5e-8, graph=True, fp32=True, guess=3),
        # the Jacobi variant of the implicit part, device-resident
        step("dplusgs_128", 128, 96, 128, its=12, solver=1),
        # the explicit path of the shipped driver, with viscous terms
        {"name": "rk3_128", "kind": "rk3", "X": 128, "Y": 96, "Z": 128, "steps": 10, "dt": 5e-9, "beta": 2.0},
        # a reference driver's inner iteration, one host-array call per function
        {"name": "host_calls_40", "kind": "host", "X": 40, "Y": 36, "Z": 40, "beta": 1.5},
        # the same driver with its limiter, filter and DPLUSGS switches on
        {"name": "host_variants_32", "kind": "variants", "X": 32, "Y": 28, "Z": 37, "beta": 1.5},
        # the training loop of the learned initial iterate on captured crops
        {"name": "train_32", "kind": "train", "crops": 256, "batch": 32, "steps": 20},
        # one loss and gradient on given crops
        {"name": "gradient_8", "kind": "gradient", "crops": 8},
    ]


def step(name, X, Y, Z, its, dt=1e-8, beta=2.0, periodic=False, graph=False, fp32=False, guess=0, order=2, solver=0):
    """One physical step of `its` inner iterations."""
    return {"name": name, "kind": "step", "X": X, "Y": Y, "Z": Z, "its": its, "dt": dt, "beta": beta,
            "periodic": periodic, "graph": graph, "fp32": fp32, "guess": guess, "order": order, "solver": solver}


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step"] * 7 + ["rk3", "host", "variants", "train", "gradient"])
    if kind == "step":
        solver = 1 if rng.random() < 0.15 else 0
        fp32 = solver == 0 and rng.random() < 0.5
        guess = rng.choice([0, 0, 1, 2]) if solver == 0 else 0
        c = step("", size(8, 224), size(8, 160), size(8, 224), its=size(2, 40), beta=rng.choice([1.5, 2.0]),
                 periodic=rng.random() < 0.3, graph=rng.random() < 0.6, fp32=fp32, guess=guess,
                 order=rng.choice([2, 3]), solver=solver)
        del c["name"]
        return c
    if kind == "rk3":
        return {"kind": "rk3", "X": size(8, 192), "Y": size(8, 128), "Z": size(8, 192), "steps": rng.randint(1, 10),
                "dt": 5e-9, "beta": rng.choice([1.5, 2.0])}
    if kind in ("host", "variants"):
        return {"kind": kind, "X": size(8, 40), "Y": size(8, 36), "Z": size(8, 64), "beta": 1.5}
    if kind == "train":
        return {"kind": "train", "crops": rng.randint(40, 256), "batch": size(4, 48), "steps": rng.randint(2, 20)}
    return {"kind": "gradient", "crops": size(1, 32)}


# --- inputs ------------------------------------------------------------------

def noisy_channel(cfg, flow, seed, thermal=0.0):
    """Laminar Poiseuille flow with 5% velocity noise on the interior, as five
    host arrays (rho, rho u, rho v, rho w, rho E); `thermal` adds noise to the
    density (the limiters divide by its differences)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape = (cfg.X_out, cfg.Y_out, cfg.Z_out)

    def noise(a):
        return (torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64) * 2 - 1) * a

    Ub, rho0 = flow.bulk_state(cfg.high)
    h = 0.5 * cfg.high
    y = torch.from_numpy(cell_y(cfg)).cuda()
    u = (1.5 * Ub * (1 - (y / h - 1) ** 2))[None, :, None] * (1 + noise(flow.noise))
    v, w = noise(flow.noise) * Ub, noise(flow.noise) * Ub
    rho = rho0 * (1 + noise(thermal)) if thermal else torch.full(shape, rho0, device="cuda", dtype=torch.float64)
    E = rho0 * R_GAS * T_WALL / (GAS - 1) + 0.5 * rho * (u * u + v * v + w * w)
    return [a.cpu().numpy() for a in (rho, rho * u, rho * v, rho * w, E)]


def channel(c, **more):
    cfg, flow = channel_cfg((c["X"], c["Y"], c["Z"]), beta=c["beta"], deltaT=c.get("dt", 1e-8), **more)
    cfg.x_periodic = c.get("periodic", False)
    return cfg, flow


def host_arrays(cfg, n=5):
    return [np.zeros((cfg.X_out, cfg.Y_out, cfg.Z_out)) for _ in range(n)]


def prepare_step(c, seed):
    # tol below any residual: every step runs its cap of inner iterations
    cfg, flow = channel(c, tol=1e-300, cap=c["its"])
    s = Solver(cfg, precision=CF_FP32_SWEEPS if c["fp32"] else CF_FP64)
    s.Jacobian_all(cfg.gamma_metric, want_arrays=False)
    s.set_implicit_solver(c["solver"])
    s.set_graph(c["graph"])
    pred = None
    if c["guess"] == 3:
        pred = Predictor(dataset_crops=1, batch_crops=1)
        load(pred, WEIGHTS / "predictor_g64x64x64_dt5e-8.npz")
        s.set_predictor(pred)
    if c["order"] == 3:
        s.set_extrapolation_order(3)
    s.set_initial_guess(c["guess"])
    Q = noisy_channel(cfg, flow, seed)
    s.load_state(Q, Q)
    if c["guess"] == 3:  # the network starts a step once three levels are known
        s.physical_step()
    return {"solver": s, "pred": pred, "Q": host_arrays(cfg)}


def run_step(st):
    s = st["solver"]
    its, er = s.physical_step()
    return {"its": its, "er": er, "Q": read_level(s, st["Q"])}


def read_level(s, Q):
    """Level n into the caller's five arrays (cf_read_state)."""
    P = ctypes.POINTER(ctypes.c_double)
    s._chk(s.lib.cf_read_state(s._h, (P * 5)(*[q.ctypes.data_as(P) for q in Q]), None, None))
    return Q


def prepare_rk3(c, seed):
    cfg, flow = channel(c)
    s = Solver(cfg)
    s.Jacobian_all(cfg.gamma_metric, want_arrays=False)
    Q = noisy_channel(cfg, flow, seed)
    s.load_state(Q, Q)
    return {"solver": s, "steps": c["steps"], "Q": host_arrays(cfg)}


def run_rk3(st):
    s = st["solver"]
    for _ in range(st["steps"]):
        s.rk3_step(viscous=True)
        s.advance_levels()
    return {"Q": read_level(s, st["Q"])}


def prepare_host(c, seed):
    """What a reference driver holds: metrics and states in its own arrays."""
    cfg, flow = channel(c)
    s = Solver(cfg)
    met = s.Jacobian_all(cfg.gamma_metric)
    Q = noisy_channel(cfg, flow, seed, thermal=0.01)
    inner = (slice(3, cfg.gend + 1), slice(2, cfg.ny + 1), slice(2, cfg.nz + 1))
    U = [np.zeros(cfg.shape) for _ in range(5)]
    for a, q in zip(U, Q):
        a[inner] = q / met["J"][inner]
    s.boundary_conditions(U, met["J"])
    st = {"solver": s, "met": met, "U_": [a.copy() for a in U], "U": U, "Uq": [a.copy() for a in U], "cfg": cfg}
    if c["kind"] == "variants":
        st["Yp"] = s.Grid(1.5)[1]
    return st


def run_host(st):
    s, m, U_ = st["solver"], st["met"], st["U_"]
    s.boundary_conditions(U_, m["J"])
    Fx = s.Flux_X(U_, m["J"], m["J_u"], m["m_u"])
    Fy = s.Flux_Y(U_, m["J"], m["J_v"], m["m_v"])
    Fz = s.Flux_Z(U_, m["J"], m["J_w"], m["m_w"])
    vF = s.Viscous_terms(U_, m)
    er, MR, NR, NL = s.Dual_time_stepping(U_, st["U"], st["Uq"], m, Fx, Fy, Fz, vF)
    return {"F": Fx + Fy + Fz, "vF": vF, "er": er, "MR": MR, "NR": NR, "NL": NL, "U_": U_}


def run_variants(st):
    s, m, U_, cfg = st["solver"], st["met"], st["U_"], st["cfg"]
    s.boundary_conditions(U_, m["J"])
    Ep = s.Filter(cfg.Roe_criterion, cfg.E_high, cfg.E_low, U_, st["Yp"], m["J"])
    Fx = s.Flux_X_limiter(U_, m["J"], m["J_u"], m["m_u"], Ep[0])
    Fy = s.Flux_Y_limiter(U_, m["J"], m["J_v"], m["m_v"], Ep[1])
    Fz = s.Flux_Z_limiter(U_, m["J"], m["J_w"], m["m_w"], Ep[2])
    vF = s.Viscous_terms(U_, m)
    er, MR, NR, NL = s.DPLUSGS(U_, st["U"], st["Uq"], m, Fx, Fy, Fz, vF)
    return {"Ep": Ep, "F": Fx + Fy + Fz, "vF": vF, "er": er, "MR": MR, "NR": NR, "NL": NL, "U_": U_}


def prepare_train(c, seed):
    """Crops of a short run's physical steps, as the training script takes them."""
    cfg, flow = channel({"X": 32, "Y": 32, "Z": 32, "beta": 2.0}, tol=1e-300, cap=12)
    Q = noisy_channel(cfg, flow, seed)
    p = Predictor(dataset_crops=c["crops"], batch_crops=c["batch"])
    with Solver(cfg) as s:
        s.Jacobian_all(cfg.gamma_metric, want_arrays=False)
        s.keep_levels(4)
        s.load_state(Q, Q)
        for _ in range(3):
            s.physical_step()
        p.capture(s, c["crops"], seed=seed)
    p.fit_norm()
    p.init_params(seed)
    return {"pred": p, "n": c["crops"], "steps": c["steps"], "seed": seed}


def run_train(st):
    p = st["pred"]
    losses = p.train(st["n"], steps=st["steps"], lr=1e-3, seed=st["seed"])
    return {"losses": losses, "params": p.get_params()}


def gradient_inputs(c, seed):
    """Crops of normalised features and targets, and He-style weights."""
    r = np.random.default_rng(seed)
    n = c["crops"]
    x = r.standard_normal((n, 16, 16, 16, 16), dtype=np.float32)
    x[..., 15] = 1.0
    t = r.standard_normal((n, 14, 14, 14, 5), dtype=np.float32)
    parts = [r.standard_normal(64 * 16) / 4, r.standard_normal(27 * 64 * 64) * math.sqrt(2 / (27 * 64)),
             r.standard_normal(64) * 0.1, r.standard_normal(5 * 64) * 0.2, r.standard_normal(5) * 0.1]
    return x, t, np.concatenate(parts).astype(np.float32)


def prepare_gradient(c, seed):
    x, t, params = gradient_inputs(c, seed)
    p = Predictor(dataset_crops=1, batch_crops=c["crops"])
    p.set_params(params)
    return {"pred": p, "x": x, "t": t}


def run_gradient(st):
    g, loss = st["pred"].gradient(st["x"], st["t"])
    return {"gradient": g, "loss": loss}


PREPARE = {"step": prepare_step, "rk3": prepare_rk3, "host": prepare_host, "variants": prepare_host,
           "train": prepare_train, "gradient": prepare_gradient}
RUN = {"step": run_step, "rk3": run_rk3, "host": run_host, "variants": run_variants, "train": run_train,
       "gradient": run_gradient}


def prepare(case, seed):
    st = PREPARE[case["kind"]](case, seed)
    st["run"] = RUN[case["kind"]]
    return st


def run(state):
    return state["run"](state)


# --- what a pass cannot do without --------------------------------------------

# FP64 operations per cell, counted from the formulas: three face fluxes of two
# reconstructions and a Roe flux each, the viscous faces, the right-hand side
# with its transform, the two triangular sweeps, the primitive update
FLUX, VISC, RHS, SWEEPS, UPDATE, JACOBI, RK = 1000, 310, 150, 290, 50, 2400, 60
# multiply-adds of the network per cell: 16 -> 64, 27 taps of 64 -> 64, 64 -> 5
NET = 64 * 16 + 27 * 64 * 64 + 64 * 5


def work(case):
    k = case["kind"]
    if k in ("train", "gradient"):
        n = case["batch"] * case["steps"] if k == "train" else case["crops"]
        cell = 24 if k == "train" else 16 + 5  # floats read per cell of a crop
        params = CF_PRED_NPARAM * 4 * (8 * case["steps"] if k == "train" else 2)  # p, m, v, g in and out
        # forward, the gradient to the weights and the gradient to h1
        return {"bytes": n * 16 ** 3 * cell * 4 + params, "flops": 3 * 2 * NET * n * 14 ** 3}
    cells = case["X"] * case["Y"] * case["Z"]
    if k == "step":
        solve = JACOBI if case["solver"] else SWEEPS
        # U_, U^n, U^{n-1} in and U_ out per iteration; the level read at the end
        return {"bytes": cells * 8 * (20 * case["its"] + 5),
                "flops": cells * case["its"] * (FLUX + VISC + RHS + solve + UPDATE)}
    if k == "rk3":
        return {"bytes": cells * 8 * (15 * 3 * case["steps"] + 5),
                "flops": cells * 3 * case["steps"] * (FLUX + VISC + RK)}
    # host calls: the states and metrics in, the fluxes, terms, increments and
    # the state out
    fields = 15 + 40 + 15 + 4 + 15 + 5
    return {"bytes": cells * 8 * fields,
            "flops": cells * (FLUX + VISC + RHS + (JACOBI if k == "variants" else SWEEPS) + UPDATE)}


def exact(case, seed):
    """The gradient in 64 bits.  The solver's own arithmetic is 64-bit IEEE
    throughout, each operation as the reference orders it, and a training run
    amplifies every rounding, so neither has a value closer than the one it
    returns."""
    if case["kind"] != "gradient":
        return None
    x, t, flat = gradient_inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = torch.from_numpy(flat).to(dev, torch.float64).requires_grad_(True)
    W1, W2, b2, W3, b3 = torch.split(p, [64 * 16, 27 * 64 * 64, 64, 5 * 64, 5])
    xs, ts = torch.from_numpy(x).to(dev, torch.float64), torch.from_numpy(t).to(dev, torch.float64)
    h = xs.reshape(-1, 16) @ W1.reshape(64, 16).t()
    h = h.reshape(-1, 16, 16, 16, 64)
    taps = W2.reshape(27, 64, 64)
    z = b2
    for q in range(27):
        i, j, l = q // 9, q // 3 % 3, q % 3
        z = z + (h[:, i:i + 14, j:j + 14, l:l + 14].reshape(-1, 64) @ taps[q].t())
    a = 0.5 * z * (1 + torch.erf(z / math.sqrt(2)))
    y = a @ W3.reshape(5, 64).t() + b3
    loss = ((y - ts.reshape(-1, 5)) ** 2).mean()
    loss.backward()
    return {"gradient": p.grad.cpu().numpy(), "loss": loss.item()}
