"""The framework's work as its users have it done, case by case, for timing.

Every case goes through the package's public entry points, on the sizes of the
reference's own experiments (20x30 Couette, 300x300 shear wave, 420x180
channel), of this repository's configurations and benchmark (4200x1800 and
8192x2048 channels, 2048x2048 boxes, uneven batches of channels) and on odd
sizes between them.  A case is a dict of plain values; its ``kind`` says which
entry points it takes:

``ops``    the four stateless drop-ins on device tensors, in the order a
           hand-written loop calls them: streaming, density, velocity field,
           equilibrium.
``step``   ``steps`` calls of ``lattice_boltzmann_step``, each fed with the
           result of the last, on device tensors or (``host``) numpy arrays.
``run``    one simulation on a ``Lattice``: load the initial moments, ``steps``
           steps, read the final fields; with ``snap`` a |u| snapshot every
           ``snap`` steps and with ``probe`` the velocity trace of one node.
           ``temporal`` is the steps-per-launch setting (0: as constructed).
``batch``  ``jobs`` uneven channels advanced together by a ``Batch``.
"""

import math
import random

import numpy as np
import torch

from lattice_boltzmann_parallel_solver_amd import Batch, Lattice
from lattice_boltzmann_parallel_solver_amd import boundary_utils as bu
from lattice_boltzmann_parallel_solver_amd import lattice_boltzmann_method as lbm
from lattice_boltzmann_parallel_solver_amd import workloads

# D2Q9 of the reference: rest, E, N, W, S, NE, NW, SW, SE
CX = (0, 1, 0, -1, 0, 1, -1, -1, 1)
CY = (0, 0, 1, 0, -1, 1, 1, -1, -1)
OPP = (0, 3, 4, 1, 2, 7, 8, 5, 6)
W = (4 / 9,) + (1 / 9,) * 4 + (1 / 36,) * 4
U_IN = 0.1      # channel inlet
U_WALL = 0.05   # Couette wall
DP = 0.001      # Poiseuille pressure difference around 1/3

# node steps of the largest listed case; drawn cases stay below a part of it
LARGEST = 8192 * 2048 * 200


def listed():
    return [
        # the reference's Couette example, one call at a time: latency only
        dict(name="step_couette_20x30", kind="step", lx=20, ly=30, bc="couette", steps=10, host=False, omega=1.0),
        # imports swapped and nothing else: the 420x180 channel on numpy arrays
        dict(name="step_numpy_channel_420x180", kind="step", lx=420, ly=180, bc="channel", steps=4, host=True,
             omega=1.6),
        # the same loop on device tensors at the large channel's size
        dict(name="step_channel_4200x1800", kind="step", lx=4200, ly=1800, bc="channel_walls", steps=3, host=False,
             omega=1 / 1.7),
        # a hand-written loop of the stateless drop-ins: odd size in FP32, and the large channel in FP64
        dict(name="ops_f32_1021x773", kind="ops", lx=1021, ly=773, dtype="f32"),
        dict(name="ops_f64_4200x1800", kind="ops", lx=4200, ly=1800, dtype="f64"),
        # shear wave decay, the lattice used as constructed
        dict(name="run_shear_300x300_f64", kind="run", lx=300, ly=300, bc="periodic", storage="f64", temporal=0,
             steps=600, omega=1.2, probe=False, snap=0),
        # the reference's vortex-street experiment: velocity probe every step, |u| snapshots, two steps per launch
        dict(name="run_channel_420x180_f64", kind="run", lx=420, ly=180, bc="channel", storage="f64", temporal=2,
             steps=600, omega=1 / 0.62, probe=True, snap=200),
        # pressure-driven box, as constructed (two steps per launch are refused there)
        dict(name="run_poiseuille_2048x2048_f64", kind="run", lx=2048, ly=2048, bc="poiseuille", storage="f64",
             temporal=0, steps=60, omega=1.5, probe=False, snap=0),
        # the large channel in the reference's precision
        dict(name="run_channel_4200x1800_f64", kind="run", lx=4200, ly=1800, bc="channel_walls", storage="f64",
             temporal=2, steps=100, omega=1 / 1.7, probe=True, snap=0),
        # the benchmark channel in FP32
        dict(name="run_channel_8192x2048_f32", kind="run", lx=8192, ly=2048, bc="channel_walls", storage="f32",
             temporal=2, steps=200, omega=1 / 1.7, probe=False, snap=0),
        # an odd Couette box in FP16 storage
        dict(name="run_couette_1531x1023_f16", kind="run", lx=1531, ly=1023, bc="couette", storage="f16", temporal=2,
             steps=200, omega=1.0, probe=False, snap=0),
        # a parameter sweep: uneven channels in one batch, the setting the server uses
        dict(name="batch_20_channels_f32", kind="batch", jobs=20, draw_seed=3, storage="f32", temporal=3, steps=121),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["ops", "step", "run", "run", "run", "run", "batch"])
    if kind == "ops":
        return dict(kind="ops", lx=_log(rng, 16, 4200), ly=_log(rng, 16, 2048), dtype=rng.choice(["f64", "f32"]))
    bc = rng.choice(["periodic", "couette", "poiseuille", "channel", "channel_walls", "channel_walls"])
    omega = round(rng.uniform(0.6, 1.7), 3)
    if kind == "step":
        host = rng.random() < 0.3
        lx, ly = (_log(rng, 20, 420), _log(rng, 30, 300)) if host else (_log(rng, 20, 4200), _log(rng, 30, 2048))
        return dict(kind="step", lx=lx, ly=ly, bc=bc, steps=rng.randint(1, 6), host=host, omega=omega)
    if kind == "batch":
        return dict(kind="batch", jobs=rng.randint(2, 20), draw_seed=rng.randrange(1000),
                    storage=rng.choice(["f32", "f32", "f64"]), temporal=rng.choice([1, 2, 3]),
                    steps=_log(rng, 20, 200))
    lx, ly = _log(rng, 48, 8192), _log(rng, 32, 2048)
    storage = rng.choice(["f64", "f64", "f32", "f32", "f16"])
    allowed = [0] if bc == "poiseuille" else [0, 2, 2]
    if bc != "poiseuille" and storage != "f64" and ly <= 1024:
        allowed.append(3)
    steps = _log(rng, 16, 800)
    steps = max(8, min(steps, LARGEST // 4 // (lx * ly)))
    return dict(kind="run", lx=lx, ly=ly, bc=bc, storage=storage, temporal=rng.choice(allowed), steps=steps,
                omega=omega, probe=rng.random() < 0.5, snap=0 if rng.random() < 0.7 else max(1, steps // 3))


# ----------------------------------------------------------------- inputs
def _plate(ly):
    return max(2, 2 * (ly // 9))


def _boundary(bc, lx, ly):
    if bc == "periodic":
        return None
    if bc == "couette":
        return bu.couette_flow_boundary_conditions(lx, ly, U_WALL, 1.0)
    if bc == "poiseuille":
        return bu.poiseuille_flow_boundary_conditions(lx, ly, (1 + DP) / 3, (1 - DP) / 3)
    walls = bc == "channel_walls"
    return bu.von_karman_boundary_conditions(lx, ly, 1.0, U_IN, _plate(ly), walls=walls, y_offset=1 if walls else 0)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _moments(lx, ly, bc, seed):
    """Density near 1 and the flow the boundary drives, with a few smooth waves
    on both (amplitudes 0.4 % and 0.01), float64."""
    rs = np.random.default_rng([seed, lx, ly])
    dev = _device()
    x = torch.arange(lx, dtype=torch.float64, device=dev)[:, None] * (2 * math.pi / lx)
    y = torch.arange(ly, dtype=torch.float64, device=dev)[None, :] * (2 * math.pi / ly)
    rho = torch.ones((lx, ly), dtype=torch.float64, device=dev)
    u = torch.zeros((lx, ly, 2), dtype=torch.float64, device=dev)
    if bc.startswith("channel"):
        u[..., 0] = U_IN
    elif bc == "periodic":
        u[..., 0] = 0.05 * torch.sin(y)
    for _ in range(3):
        kx, ky = (int(k) for k in rs.integers(1, 4, 2))
        a, b, c = rs.uniform(0, 2 * math.pi, 3)
        amp = rs.uniform(0.3, 1.0, 3)
        rho += 0.0013 * amp[0] * torch.sin(kx * x + a) * torch.cos(ky * y + b)
        u[..., 0] += 0.0033 * amp[1] * torch.cos(kx * x + b) * torch.sin(ky * y + c)
        u[..., 1] += 0.0033 * amp[2] * torch.sin(kx * x + c) * torch.cos(ky * y + a)
    return rho, u


def _step_input(case, seed):
    """Populations a little off the equilibrium of the moments, and their own moments."""
    lx, ly = case["lx"], case["ly"]
    rho, u = _moments(lx, ly, case.get("bc", "periodic"), seed)
    f = _equilibrium(rho, u)
    x = torch.arange(lx, dtype=torch.float64, device=f.device)[:, None] * 0.7
    y = torch.arange(ly, dtype=torch.float64, device=f.device)[None, :] * 0.3
    for i in range(9):
        f[..., i] *= 1 + 0.002 * torch.sin(x * (i + 1) + y + seed % 7)
    rho = f.sum(-1)
    return f, rho, _velocity(rho, f)


def _jobs(case):
    return workloads.channel_jobs(case["jobs"], seed=case["draw_seed"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ops":
        f, _, _ = _step_input(case, seed)
        return dict(case=case, f=f.to(torch.float32) if case["dtype"] == "f32" else f)
    if kind == "step":
        ins = _step_input(case, seed)
        if case["host"]:
            ins = tuple(t.cpu().numpy() for t in ins)
        return dict(case=case, ins=ins, boundary=_boundary(case["bc"], case["lx"], case["ly"]))
    if kind == "run":
        lx, ly = case["lx"], case["ly"]
        lat = Lattice(lx, ly, boundary=_boundary(case["bc"], lx, ly), storage=case["storage"])
        if case["temporal"]:
            lat.set_temporal(case["temporal"])
        if case["probe"]:
            lat.set_probe(3 * lx // 4, ly // 2, case["steps"])
        return dict(case=case, lat=lat, init=_moments(lx, ly, case["bc"], seed), out=_outputs(lx, ly))
    lats, inits, outs = [], [], []
    jobs = _jobs(case)
    for k, job in enumerate(jobs):
        lats.append(workloads.build_lattice(job, case["storage"]))
        inits.append(_moments(job.lx, job.ly, "channel_walls", seed + 1000 * k))
        outs.append(_outputs(job.lx, job.ly))
    batch = Batch(lats, [job.omega for job in jobs], temporal=case["temporal"])
    return dict(case=case, lats=lats, batch=batch, inits=inits, outs=outs)


def _outputs(lx, ly):
    return tuple(torch.empty(s, dtype=torch.float64, device="cuda") for s in ((lx, ly, 9), (lx, ly), (lx, ly, 2)))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ops":
        f = lbm.streaming(state["f"])
        rho = lbm.compute_density(f)
        u = lbm.compute_velocity_field(rho, f)
        return f, rho, u, lbm.equilibrium_distr_func(rho, u)
    if kind == "step":
        f, rho, u = state["ins"]
        for _ in range(case["steps"]):
            f, rho, u = lbm.lattice_boltzmann_step(f, rho, u, case["omega"], state["boundary"])
        return f, rho, u
    if kind == "run":
        lat, steps, snap = state["lat"], case["steps"], case["snap"]
        lat.set_equilibrium(*state["init"])
        result = {}
        if snap:
            speeds = []
            for _ in range(steps // snap):
                lat.run(case["omega"], snap)
                speeds.append(lat.speed())
            lat.run(case["omega"], steps % snap)
            result["speed"] = speeds
        else:
            lat.run(case["omega"], steps)
        lat.state_into(*state["out"])
        if case["probe"]:
            result["probe"] = lat.probe()
        result["f"], result["rho"], result["u"] = state["out"]
        return result
    for lat, init in zip(state["lats"], state["inits"]):
        lat.set_equilibrium(*init)
    state["batch"].run(case["steps"])
    for lat, out in zip(state["lats"], state["outs"]):
        lat.state_into(*out)
    return state["outs"]


def work(case):
    """Inputs read once and outputs written once; about 130 operations per node
    and step (moments 18, velocity 2, equilibrium 83, relaxation 27)."""
    kind = case["kind"]
    if kind == "batch":
        n = sum(job.nodes for job in _jobs(case))
        return {"bytes": n * (3 + 12) * 8, "flops": n * case["steps"] * 130}
    n = case["lx"] * case["ly"]
    if kind == "ops":
        # f in; f, rho, u and the equilibrium out
        return {"bytes": n * (9 + 9 + 1 + 2 + 9) * (4 if case["dtype"] == "f32" else 8), "flops": n * 103}
    if kind == "step":
        # each call takes (f, rho, u) and gives (f, rho, u)
        return {"bytes": n * 24 * 8 * case["steps"], "flops": n * case["steps"] * 130}
    bytes_ = n * (3 + 12) * 8
    if case["snap"]:
        bytes_ += n * 8 * (case["steps"] // case["snap"])
    if case["probe"]:
        bytes_ += 24 * case["steps"]
    return {"bytes": bytes_, "flops": n * case["steps"] * 130}


# ----------------------------------------------------- plain 64-bit reference
def _equilibrium(rho, u):
    ux, uy = u[..., 0], u[..., 1]
    usq = 1.5 * (ux * ux + uy * uy)
    out = torch.empty(rho.shape + (9,), dtype=rho.dtype, device=rho.device)
    for i in range(9):
        cu = CX[i] * ux + CY[i] * uy
        out[..., i] = W[i] * rho * (1 + 3 * cu + 4.5 * cu * cu - usq)
    return out


def _velocity(rho, f):
    return torch.stack([(f[..., 1] + f[..., 5] + f[..., 8] - f[..., 3] - f[..., 6] - f[..., 7]) / rho,
                        (f[..., 2] + f[..., 5] + f[..., 6] - f[..., 4] - f[..., 7] - f[..., 8]) / rho], dim=-1)


def _stream(f):
    return torch.stack([torch.roll(f[..., i], (CX[i], CY[i]), (0, 1)) for i in range(9)], dim=-1)


def _reflect(pre, post, where, dirs, k=None):
    for i in dirs:
        post[where + (OPP[i],)] = pre[where + (i,)] - (k[i] if k else 0.0)


def _step(f, rho, u, omega, bc, plate):
    """collide with (rho, u), stream, boundary, moments."""
    lx, ly = rho.shape
    feq = _equilibrium(rho, u)
    pre = f + omega * (feq - f)
    if bc == "poiseuille":
        ones = torch.ones(ly, dtype=f.dtype, device=f.device)
        e_in = _equilibrium(ones * (1 + DP), u[-2])
        e_out = _equilibrium(ones * (1 - DP), u[1])
        new0 = e_in + (pre[-2] - feq[-2])
        new1 = e_out + (pre[1] - feq[1])
        for i in (1, 5, 8):
            pre[0, :, i] = new0[:, i]
        for i in (3, 6, 7):
            pre[-1, :, i] = new1[:, i]
    post = _stream(pre)
    full = slice(None)
    if bc == "couette":
        _reflect(pre, post, (full, ly - 1), (2, 5, 6))
        k = [6 * W[i] * CX[i] * U_WALL for i in range(9)]
        _reflect(pre, post, (full, 0), (4, 7, 8), k)
    elif bc == "poiseuille":
        _reflect(pre, post, (full, 0), (4, 7, 8))
        _reflect(pre, post, (full, ly - 1), (2, 5, 6))
    elif bc.startswith("channel"):
        x = lx // 4
        y0 = ly // 2 - plate // 2 + (1 if bc == "channel_walls" else 0)
        y1 = y0 + 2 * (plate // 2) - 1
        inlet = torch.tensor([1.0, U_IN, 0.0], dtype=f.dtype, device=f.device)
        post[0] = _equilibrium(inlet[:1], inlet[None, 1:])
        for i in (3, 6, 7):
            post[-1, :, i] = f[-2, :, i]
        _reflect(pre, post, (x, slice(y0 + 1, y1)), (1, 5, 8))
        _reflect(pre, post, (x + 1, slice(y0 + 1, y1)), (3, 6, 7))
        # two-cell plates have no interior: only their corners act
        _reflect(pre, post, (x + 1, slice(y1, y1 + 1)), (3, 7))
        _reflect(pre, post, (x + 1, slice(y0, y0 + 1)), (3, 6))
        _reflect(pre, post, (x, slice(y1, y1 + 1)), (1, 8))
        _reflect(pre, post, (x, slice(y0, y0 + 1)), (1, 5))
        if bc == "channel_walls":
            _reflect(pre, post, (full, 0), (4, 7, 8))
            _reflect(pre, post, (full, ly - 1), (2, 5, 6))
    rho = post.sum(-1)
    return post, rho, _velocity(rho, post)


def _simulate(init, case, plate, omega, bc):
    lx, ly = init[0].shape
    rho, u = init
    f = _equilibrium(rho, u)
    speeds, probe = [], []
    for n in range(1, case["steps"] + 1):
        f, rho, u = _step(f, rho, u, omega, bc, plate)
        if case.get("snap") and n % case["snap"] == 0:
            speeds.append((u[..., 0] ** 2 + u[..., 1] ** 2).sqrt().cpu().numpy())
        if case.get("probe"):
            probe.append(torch.cat([rho[3 * lx // 4, ly // 2][None], u[3 * lx // 4, ly // 2]]))
    return f, rho, u, speeds, probe


def exact(case, seed):
    kind = case["kind"]
    if kind == "ops":
        f, _, _ = _step_input(case, seed)
        if case["dtype"] == "f32":
            f = f.to(torch.float32).to(torch.float64)
        f = _stream(f)
        rho = f.sum(-1)
        u = _velocity(rho, f)
        return f, rho, u, _equilibrium(rho, u)
    if kind == "step":
        f, rho, u = _step_input(case, seed)
        for _ in range(case["steps"]):
            f, rho, u = _step(f, rho, u, case["omega"], case["bc"], _plate(case["ly"]))
        return tuple(t.cpu().numpy() for t in (f, rho, u)) if case["host"] else (f, rho, u)
    if kind == "run":
        init = _moments(case["lx"], case["ly"], case["bc"], seed)
        f, rho, u, speeds, probe = _simulate(init, case, _plate(case["ly"]), case["omega"], case["bc"])
        result = {"f": f, "rho": rho, "u": u}
        if case["snap"]:
            result["speed"] = speeds
        if case["probe"]:
            result["probe"] = torch.stack(probe).cpu().numpy()
        return result
    outs = []
    for k, job in enumerate(_jobs(case)):
        init = _moments(job.lx, job.ly, "channel_walls", seed + 1000 * k)
        outs.append(_simulate(init, case, job.plate, job.omega, "channel_walls")[:3])
    return outs
