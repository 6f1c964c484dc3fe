"""Performance cases: the work a user of azeban_amd has it do, through its public entry points.

Time stepping dominates every use, so most cases are steps of the solver: single small
grids (latency), the benchmark grids (2D 1024^2, 3D 512^3), batched ensembles, in FP64 and
in FP32-mixed.  The others are what surrounds the stepping: initial data from physical
space, physical output with its energy spectrum, and the standalone transforms.

Inputs are double shear layers (2D) and fractional-Brownian velocity fields (3D), made on
the GPU from the seed; exact() recomputes every result with torch's transforms in 64 bits.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import azeban_amd as A
from azeban_amd.ensemble import Ensemble, Group

CFL = 0.2
T_FAR = 1e6  # target time that no case reaches: the step count ends the call

PRECISIONS = ("fp64", "fp32_mixed")
SOLVER_2D = (64, 128, 256, 512, 1024)
SOLVER_3D = (64, 128, 256, 512)
# transform lengths (powers of two and three times them)
LENGTHS = (48, 64, 96, 128, 192, 256, 384, 512, 768, 1024)


def listed() -> list:
    return [
        # one step of the smallest grid, dt returned to the caller: launches and latency
        {"name": "step_2d_64", "kind": "step", "dim": 2, "N": 64, "precision": "fp64"},
        # a short run of a small 2D sample in FP32-mixed, two host checks
        {"name": "run_2d_256_mixed", "kind": "run", "dim": 2, "N": 256, "precision": "fp32_mixed", "steps": 16},
        # the 2D benchmark: double shear layer at 1024^2
        {"name": "run_2d_1024", "kind": "run", "dim": 2, "N": 1024, "precision": "fp64", "steps": 8},
        # one step of a small 3D request
        {"name": "step_3d_64", "kind": "step", "dim": 3, "N": 64, "precision": "fp64"},
        # a run of a mid-size 3D sample in FP32-mixed
        {"name": "run_3d_128_mixed", "kind": "run", "dim": 3, "N": 128, "precision": "fp32_mixed", "steps": 8},
        # one step of the largest 3D size the solve server takes
        {"name": "step_3d_256", "kind": "step", "dim": 3, "N": 256, "precision": "fp64"},
        # the headline benchmark: one SSP-RK3 step at 512^3
        {"name": "step_3d_512", "kind": "step", "dim": 3, "N": 512, "precision": "fp64"},
        # the right-hand side alone at 512^3 in FP32-mixed (a caller with its own integrator)
        {"name": "rhs_3d_512_mixed", "kind": "rhs", "dim": 3, "N": 512, "precision": "fp32_mixed"},
        # a statistical ensemble of uneven 2D grid sizes, every sample in one graph
        {"name": "ensemble_2d", "kind": "ensemble", "n128": 33, "n256": 21, "n512": 13, "precision": "fp64",
         "steps": 8},
        # initial data of a 3D run: physical field to a divergence-free spectrum
        {"name": "init_3d_256", "kind": "init", "dim": 3, "N": 256},
        # one output time of a 3D run: the physical field and the energy spectrum
        {"name": "snapshot_3d_256", "kind": "snapshot", "dim": 3, "N": 256, "N_out": 256},
        # the standalone inverse transform in single precision, a ragged batch of 3 * 2^k lines
        {"name": "fft_c2r_2d_384_f32", "kind": "fft", "dim": 2, "N": 384, "howmany": 13, "precision": "fp32_mixed",
         "inverse": True},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["step", "run", "run", "rhs", "ensemble", "init", "snapshot", "fft"])
    if kind in ("step", "run", "rhs"):
        dim = rng.choice([2, 3])
        N = rng.choice(SOLVER_2D if dim == 2 else SOLVER_3D)
        case = {"kind": kind, "dim": dim, "N": N, "precision": rng.choice(PRECISIONS)}
        if kind == "run":
            # no more grid point steps than one step at 512^3
            case["steps"] = _log_int(rng, 1, max(1, min(24, 512**3 // N**dim // (2 if N == 256 else 1))))
        return case
    if kind == "ensemble":
        return {"kind": "ensemble", "n128": _log_int(rng, 1, 96), "n256": _log_int(rng, 1, 48),
                "n512": _log_int(rng, 1, 24), "precision": rng.choice(PRECISIONS), "steps": rng.choice([3, 4, 7, 8, 16])}
    dim = rng.choice([2, 3])
    if kind == "init":
        return {"kind": "init", "dim": dim, "N": rng.choice([n for n in LENGTHS if dim == 2 or n <= 384])}
    if kind == "snapshot":
        N = rng.choice([n for n in LENGTHS if dim == 2 or n <= 384])
        smaller = [n for n in LENGTHS if n < N]
        return {"kind": "snapshot", "dim": dim, "N": N,
                "N_out": rng.choice(smaller) if smaller and rng.random() < 0.3 else N}
    dim = rng.choice([1, 2, 3])
    N = rng.choice([n for n in LENGTHS if dim < 3 or n <= 256])
    return {"kind": "fft", "dim": dim, "N": N, "howmany": _log_int(rng, 1, max(1, min(4096, 2**25 // N**dim))),
            "precision": rng.choice(PRECISIONS), "inverse": rng.random() < 0.5}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device() -> str:
    return "cuda" if torch.cuda.is_available() else "cpu"


def _wavenumbers(dim: int, N: int):
    """2 pi times the signed mode numbers per axis, index N/2 counted as +N/2."""
    i = torch.arange(N, device=_device(), dtype=torch.float64)
    full = torch.where(i >= N // 2 + 1, i - N, i) * (2 * math.pi)
    half = torch.arange(N // 2 + 1, device=_device(), dtype=torch.float64) * (2 * math.pi)
    axes = [full] * (dim - 1) + [half]
    return [a.reshape([-1 if d == e else 1 for e in range(dim)]) for d, a in enumerate(axes)]


def _leray(u: torch.Tensor) -> torch.Tensor:
    """(1 - k k^T / |k|^2) u_hat, zero at k = 0."""
    dim = u.dim() - 1
    k = _wavenumbers(dim, u.shape[1])
    k2 = sum(x * x for x in k)
    k2.view(-1)[0] = 1.0
    kdotu = sum(k[d] * u[d] for d in range(dim)) / k2
    out = torch.stack([u[d] - k[d] * kdotu for d in range(dim)])
    out.view(dim, -1)[:, 0] = 0
    return out


def _shear_layer(N: int, seed: int, rho: float = 0.05, delta: float = 0.05) -> torch.Tensor:
    """Double shear layer with ten random sine modes on the cross-stream velocity."""
    r = random.Random(seed)
    x = torch.arange(N, device=_device(), dtype=torch.float64) / N
    X, Y = x.reshape(-1, 1), x.reshape(1, -1)
    u = torch.where(Y <= 0.5, torch.tanh((Y - 0.25) / rho), torch.tanh((0.75 - Y) / rho)).expand(N, N)
    v = delta * torch.sin(2 * math.pi * X)
    for m in range(1, 11):
        v = v + r.uniform(-0.025, 0.025) * torch.sin(2 * math.pi * m * X + r.uniform(0, 2 * math.pi))
    return torch.stack([u, v.expand(N, N)])


def _brownian_spectrum(dim: int, N: int, seed: int, hurst: float = 0.75) -> torch.Tensor:
    """Spectrum of a random field with |c_k| ~ |k|^-(H + d/2), unit RMS speed on the grid."""
    g = torch.Generator(device=_device()).manual_seed(seed)
    k = _wavenumbers(dim, N)
    k2 = sum(x * x for x in k)
    k2.view(-1)[0] = 1.0
    amp = k2.pow(-(hurst + dim / 2) / 2)
    amp.view(-1)[0] = 0.0
    comps = []
    for _ in range(dim):
        noise = torch.randn((N,) * dim, device=_device(), dtype=torch.float64, generator=g)
        c = torch.fft.rfftn(noise)
        c *= amp
        comps.append(c)
        del noise
    u = torch.stack(comps)
    # mean square speed from Parseval's sum over the half spectrum, edge columns counted once
    e = u.real.square().sum(0) + u.imag.square().sum(0)
    total = 2 * e.sum() - e[..., 0].sum() - e[..., -1].sum()
    return u * (float(N) ** dim / torch.sqrt(total))


def _physical(dim: int, N: int, seed: int) -> torch.Tensor:
    if dim == 2:
        return _shear_layer(N, seed)
    c = _brownian_spectrum(dim, N, seed)
    return torch.stack([torch.fft.irfftn(x, s=(N,) * dim) for x in c])


def _state(dim: int, N: int, seed: int) -> torch.Tensor:
    """A divergence-free Fourier state (dim, N, ..., N/2+1)."""
    if dim == 2:
        return _leray(torch.fft.rfftn(_shear_layer(N, seed), dim=(1, 2)))
    return _leray(_brownian_spectrum(dim, N, seed))


def _visc(N: int) -> A.SmoothCutoff1D:
    return A.SmoothCutoff1D(0.05 / N, 1.0, 2 * math.pi * N / 4)


def _max_dt(N: int) -> float:
    return CFL * 2.0 / (0.05 / N * (math.pi * N) ** 2)


def _ensemble_states(case: dict, seed: int) -> list:
    """Per grid size the stacked states of its samples, each from a seed of its own."""
    out = []
    for N, count in ((128, case["n128"]), (256, case["n256"]), (512, case["n512"])):
        out.append(torch.stack([_state(2, N, 1000003 * seed + 10007 * N + s) for s in range(count)]))
    return out


def _fft_input(case: dict, seed: int) -> torch.Tensor:
    dim, N = case["dim"], case["N"]
    g = torch.Generator(device=_device()).manual_seed(seed)
    x = torch.randn((case["howmany"],) + (N,) * dim, device=_device(), dtype=torch.float64, generator=g)
    if case["inverse"]:
        x = torch.fft.rfftn(x, dim=tuple(range(1, dim + 1)))
        return x if case["precision"] == "fp64" else x.to(torch.complex64)
    return x if case["precision"] == "fp64" else x.to(torch.float32)


# ---------------------------------------------------------------------------
# preparation and the pass itself
# ---------------------------------------------------------------------------
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    state = {"case": case}
    if kind in ("step", "run", "rhs"):
        dim, N = case["dim"], case["N"]
        grid = A.Grid(dim, N)
        eq = A.IncompressibleEuler(grid, _visc(N), case["precision"])
        u = _state(dim, N, seed)
        stepper = A.SSP_RK3(grid.shape_fourier(dim), eq)
        if kind == "run":
            state["sim"] = A.Simulation(grid, CFL, stepper, u)
        else:
            state.update(eq=eq, stepper=stepper, u=u)
            if kind == "rhs":
                state["dudt"] = torch.empty_like(u)
    elif kind == "ensemble":
        groups = [Group(2, u.shape[-2], u, case["precision"]) for u in _ensemble_states(case, seed)]
        state["ensemble"] = Ensemble(groups, CFL)
    elif kind == "init":
        state["u_phys"] = _physical(case["dim"], case["N"], seed)
    elif kind == "snapshot":
        state["u"] = _state(case["dim"], case["N"], seed)
    elif kind == "fft":
        state["x"] = _fft_input(case, seed)
    else:
        raise ValueError(f"unknown kind {kind}")
    return state


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        dt = state["stepper"].integrate(T_FAR, _max_dt(case["N"]), CFL, state["u"])
        return {"u": state["u"], "dt": dt}
    if kind == "run":
        sim = state["sim"]
        before = sim.time()
        steps = sim.simulate_until(T_FAR, max_steps=case["steps"])
        return {"u": sim.u(), "elapsed": sim.time() - before, "steps": steps}
    if kind == "rhs":
        state["eq"].dudt(state["dudt"], state["u"])
        return state["dudt"]
    if kind == "ensemble":
        ens = state["ensemble"]
        before = ens.times()
        ens.run(T_FAR, steps_per_launch=case["steps"], max_launches=1)
        after = ens.times()
        return {"u": [g.u for g in ens.groups],
                "elapsed": [np.array(b) - np.array(a) for a, b in zip(before, after)]}
    if kind == "init":
        return A.initialize(state["u_phys"])
    if kind == "snapshot":
        u = state["u"]
        return {"u_phys": A.to_physical(u, case["N_out"]), "spectrum": np.array(A.energy_spectrum(u))}
    if case["inverse"]:
        return A.fft_c2r(state["x"], case["N"])
    return A.fft_r2c(state["x"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _modes(dim: int, N: int) -> float:
    return float(N) ** (dim - 1) * (N // 2 + 1)


def _fft_flops(dim: int, N: int) -> float:
    return 2.5 * float(N) ** dim * math.log2(float(N) ** dim)


def _rhs_flops(dim: int, N: int) -> float:
    """dim inverse and dim(dim+1)/2 forward real transforms on the 3N/2 grid, the products,
    and the projection and viscosity per mode."""
    M = 3 * N // 2
    products = dim * (dim + 1) // 2
    return (dim + products) * _fft_flops(dim, M) + products * float(M) ** dim + 30.0 * dim * _modes(dim, N)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("step", "run", "rhs"):
        dim, N = case["dim"], case["N"]
        evaluations = {"step": 3, "rhs": 1, "run": 3 * case.get("steps", 1)}[kind]
        return {"bytes": 2 * 16.0 * dim * _modes(dim, N), "flops": evaluations * _rhs_flops(dim, N)}
    if kind == "ensemble":
        sizes = ((128, case["n128"]), (256, case["n256"]), (512, case["n512"]))
        return {"bytes": sum(2 * 16.0 * 2 * _modes(2, N) * c for N, c in sizes),
                "flops": sum(3 * case["steps"] * c * _rhs_flops(2, N) for N, c in sizes)}
    dim, N = case["dim"], case["N"]
    if kind == "init":
        return {"bytes": dim * (8.0 * float(N) ** dim + 16.0 * _modes(dim, N)),
                "flops": dim * _fft_flops(dim, N) + 12.0 * dim * _modes(dim, N)}
    if kind == "snapshot":
        n = case["N_out"]
        return {"bytes": dim * (16.0 * _modes(dim, N) + 8.0 * float(n) ** dim),
                "flops": dim * _fft_flops(dim, n) + 6.0 * dim * _modes(dim, N)}
    size = 8.0 if case["precision"] == "fp64" else 4.0
    return {"bytes": case["howmany"] * size * (float(N) ** dim + 2 * _modes(dim, N)),
            "flops": case["howmany"] * _fft_flops(dim, N)}


# ---------------------------------------------------------------------------
# the same results from torch's transforms in 64 bits
# ---------------------------------------------------------------------------
def _inverse(c: torch.Tensor, n: int) -> torch.Tensor:
    """Unnormalised c2r of one component: complex passes over the leading axes, then the
    last axis, which ignores Im at its first and middle mode."""
    if c.dim() > 1:
        c = torch.fft.ifftn(c, dim=tuple(range(c.dim() - 1)), norm="forward")
    else:
        c = c.clone()
    edge = torch.view_as_real(c)
    edge[..., 0, 1] = 0
    edge[..., n // 2, 1] = 0
    return torch.fft.irfft(c, n=n, norm="forward")


def _resize(c: torch.Tensor, n: int) -> torch.Tensor:
    """One component moved to n modes per axis: modes kept up to the smaller half, the last
    axis compact, index N/2 of a full axis counted as positive."""
    dim, N = c.dim(), c.shape[-1] * 2 - 2
    small = min(N, n)
    h = small // 2 + 1
    keep_src = torch.cat([torch.arange(h), torch.arange(N - (small - h), N)]).to(c.device)
    keep_dst = torch.cat([torch.arange(h), torch.arange(n - (small - h), n)]).to(c.device)
    for d in range(dim - 1):
        src = c.index_select(d, keep_src)
        shape = list(src.shape)
        shape[d] = n
        c = torch.zeros(shape, dtype=src.dtype, device=src.device).index_copy_(d, keep_dst, src)
    out = torch.zeros(c.shape[:-1] + (n // 2 + 1,), dtype=c.dtype, device=c.device)
    out[..., :h] = c[..., :h]
    return out


def _rhs(u: torch.Tensor):
    """(L(u_hat), max|u|) of the dealiased right-hand side with smooth-cutoff viscosity."""
    dim, N = u.dim() - 1, u.shape[1]
    M = 3 * N // 2
    phys = [_inverse(_resize(u[c], M), M) for c in range(dim)]
    u_max = max(float(p.abs().max()) for p in phys) / float(M) ** dim
    norm = 1.0 / (float(N) ** (dim / 2) * float(M) ** (dim / 2))
    for p in phys:
        p *= norm
    k = _wavenumbers(dim, N)
    b = torch.zeros_like(u)
    for r in range(dim):
        for c in range(r + 1):
            B = _resize(torch.fft.rfftn(phys[r] * phys[c]), N)
            b[r] += 1j * k[c] * B
            if c != r:
                b[c] += 1j * k[r] * B
    v = _visc(N)
    k2 = sum(x * x for x in k)
    nu = -v.eps * k2 * -torch.expm1(-(torch.sqrt(k2) / v.k0) ** 18)
    out = nu * u - _leray(b)
    out.view(dim, -1)[:, 0] = 0
    return out, u_max


def _rk3(u: torch.Tensor, max_dt: float):
    d, u_max = _rhs(u)
    dt = min(CFL / (u.shape[1] * u_max), max_dt)
    u1 = u + dt * d
    u2 = 0.75 * u + 0.25 * (u1 + dt * _rhs(u1)[0])
    return (2.0 / 3) * (u2 + dt * _rhs(u2)[0]) + (1.0 / 3) * u, dt


def _rk3_steps(u: torch.Tensor, steps: int):
    t = 0.0
    for _ in range(steps):
        u, dt = _rk3(u, _max_dt(u.shape[1]))
        t += dt
    return u, t


def _spectrum(u: torch.Tensor) -> np.ndarray:
    """Energy per shell of the largest mode number, half-spectrum modes counted twice."""
    dim, N = u.dim() - 1, u.shape[1]
    k = [(x / (2 * math.pi)).round().long().abs() for x in _wavenumbers(dim, N)]
    shell = k[0]
    for x in k[1:]:
        shell = torch.maximum(shell, x)
    e = 0.5 * (u.real.square().sum(0) + u.imag.square().sum(0)) / float(N) ** (2 * dim)
    e[..., 1:] *= 2
    return torch.bincount(shell.reshape(-1).cpu(), weights=e.reshape(-1).cpu(), minlength=N // 2 + 1).numpy()


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "rhs":
        return _rhs(_state(case["dim"], case["N"], seed))[0]
    if kind == "step":
        u, dt = _rk3(_state(case["dim"], case["N"], seed), _max_dt(case["N"]))
        return {"u": u, "dt": dt}
    if kind == "run":
        u, t = _rk3_steps(_state(case["dim"], case["N"], seed), case["steps"])
        return {"u": u, "elapsed": t, "steps": None}
    if kind == "ensemble":
        us, ts = [], []
        for stack in _ensemble_states(case, seed):
            done = [_rk3_steps(u, case["steps"]) for u in stack]
            us.append(torch.stack([u for u, _ in done]))
            ts.append(np.array([t for _, t in done]))
        return {"u": us, "elapsed": ts}
    if kind == "init":
        u = _physical(case["dim"], case["N"], seed)
        return _leray(torch.stack([torch.fft.rfftn(c) for c in u]))
    if kind == "snapshot":
        dim, N, n = case["dim"], case["N"], case["N_out"]
        u = _state(dim, N, seed)
        return {"u_phys": torch.stack([_inverse(_resize(c, n), n) for c in u]) / float(N) ** dim,
                "spectrum": _spectrum(u)}
    x = _fft_input(case, seed)
    if case["inverse"]:
        return torch.stack([_inverse(c, case["N"]) for c in x.to(torch.complex128)])
    return torch.fft.rfftn(x.double(), dim=tuple(range(1, case["dim"] + 1)))
