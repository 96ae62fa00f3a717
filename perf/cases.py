"""The work that programs have this library do, as cases that can be timed.

Two kinds of program use it.  Some call the directional compact operators on
device fields of their own (plan_direction / apply_along! / filter_field!):
the `gradient` and `filter` cases.  The others set a problem up and let run!
advance the device state, taking the state back at output times: the `tgv`
(three-dimensional Taylor-Green flow), `shock` (two-dimensional two-gas shock /
interface with characteristic faces) and `tubes` (batches of uneven
one-dimensional shock tubes) cases.  A pass of a run! case is a number of
steps and the state's return to the host, as between two outputs of a run; the
next pass goes on from there.

Sizes: 32^3 to 256^3 is the range of the Taylor-Green benchmark and tests,
1024 x 512 (and down to 96 x 48) that of the shock / interface, 128 to 2048
points that of the tubes; operators are used on the same grids and on somewhat
larger ones.
"""
import os
import sys

import torch  # before the package: one HIP runtime serves both
import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "compactles.jl_amd"))

import compactles_hip as ch  # noqa: E402
from compactles_hip import workloads  # noqa: E402

TWO_PI = 2 * np.pi


def listed():
    return [
        # the smallest grids of the tests, closed, odd: launches and latency count
        dict(name="gradient c6 closed 33x29x31", kind="gradient", scheme="c6", nx=33, ny=29, nz=31, dtype="fp64",
             periodic=False),
        # the operator benchmark's grid: the derivative every solver step is made of
        dict(name="gradient c6 256", kind="gradient", scheme="c6", nx=256, ny=256, nz=256, dtype="fp64", periodic=True),
        # the tenth-order scheme in single precision between walls, ragged extents
        dict(name="gradient c10 fp32 250x199x180", kind="gradient", scheme="c10", nx=250, ny=199, nz=180, dtype="fp32",
             periodic=False),
        # a large single-precision field
        dict(name="gradient c6 fp32 384", kind="gradient", scheme="c6", nx=384, ny=384, nz=384, dtype="fp32",
             periodic=True),
        # smoothing a field in place, odd extents
        dict(name="filter 256x255x257", kind="filter", scheme="c8", nx=256, ny=255, nz=257, dtype="fp64",
             periodic=True),
        # the smallest flow anyone runs (a test or a parameter scan)
        dict(name="tgv 32", kind="tgv", nx=32, ny=32, nz=32, dtype="fp64", steps=40),
        # the quick start's grid
        dict(name="tgv 64", kind="tgv", nx=64, ny=64, nz=64, dtype="fp64", steps=40),
        # a box with uneven odd extents in the mixed form
        dict(name="tgv fp32 120x97x81", kind="tgv", nx=120, ny=97, nz=81, dtype="fp32", steps=40),
        # the headline benchmark, in both forms
        dict(name="tgv 256", kind="tgv", nx=256, ny=256, nz=256, dtype="fp64", steps=40),
        dict(name="tgv fp32 256", kind="tgv", nx=256, ny=256, nz=256, dtype="fp32", steps=50),
        # the shock / interface benchmark
        dict(name="shock 1024x512", kind="shock", nx=1024, ny=512, dtype="fp64", steps=60),
        # a parameter study of shock tubes of uneven length
        dict(name="tubes 512", kind="tubes", count=512, nmin=128, nmax=2048, dtype="fp64", steps=96),
    ]


def _logint(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["gradient", "gradient", "filter", "tgv", "tgv", "shock", "tubes"])
    dtype = rng.choice(["fp64", "fp64", "fp32"])
    if kind in ("gradient", "filter"):
        base = _logint(rng, 26, 320)
        n = [max(24, int(base * rng.uniform(0.7, 1.25))) for _ in range(3)]
        return dict(kind=kind, scheme=rng.choice(["c6", "c6", "c10", "c4"]) if kind == "gradient" else "c8",
                    nx=n[0], ny=n[1], nz=n[2], dtype=dtype,
                    periodic=True if kind == "filter" else rng.random() < 0.5)
    if kind == "tgv":
        base = _logint(rng, 28, 190)
        n = [max(24, int(base * rng.uniform(0.75, 1.2))) for _ in range(3)]
        if rng.random() < 0.3:
            n = [base] * 3
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], dtype=dtype, steps=rng.randint(20, 40))
    if kind == "shock":
        nx = _logint(rng, 96, 1024)
        return dict(kind=kind, nx=nx, ny=max(48, int(nx * rng.uniform(0.4, 0.6))), dtype=dtype,
                    steps=rng.randint(30, 60))
    return dict(kind=kind, count=_logint(rng, 32, 512), nmin=128, nmax=rng.randint(512, 2048), dtype=dtype,
                steps=rng.randint(48, 96))


def _n(case):
    return case["nx"], case["ny"], case["nz"]


def _real(case):
    return torch.float64 if case["dtype"] == "fp64" else torch.float32


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
def _smooth_field(case, seed):
    """A smooth turbulence-like field (a few dozen Fourier modes, decaying
    amplitudes) as a float64 tensor of shape (nz, ny, nx) on the GPU."""
    n = _n(case)
    g = np.random.default_rng(seed)
    # periodic grids leave out the end point, closed ones hold both ends
    x = [torch.arange(m, dtype=torch.float64, device="cuda") * (TWO_PI / (m if case["periodic"] else m - 1)) for m in n]
    f = torch.zeros(n[::-1], dtype=torch.float64, device="cuda")
    for _ in range(24):
        k = g.integers(0, 9, 3)
        ph = g.uniform(0, TWO_PI, 3)
        amp = g.standard_normal() / (1 + float(k @ k)) ** (5 / 6)
        cx, cy, cz = (torch.cos(int(k[d]) * x[d] + ph[d]) for d in range(3))
        f += amp * cz[:, None, None] * cy[None, :, None] * cx[None, None, :]
    return f


class _CudaArray:
    """A DeviceArray as the array interface torch reads (no copy)."""

    def __init__(self, a):
        self.keep = a
        self.__cuda_array_interface__ = {"shape": a.shape[::-1], "typestr": a.dtype.str, "version": 3,
                                         "data": (a.ptr.value, False), "strides": None}


def _interior(a, decomp):
    """The interior of a padded DeviceArray as a torch view, x fastest."""
    t = torch.as_tensor(_CudaArray(a), device="cuda")
    hx, hy, hz = decomp.n_halo_d
    nx, ny, nz = decomp.n_local
    return t[hz:hz + nz, hy:hy + ny, hx:hx + nx]


def _tgv_state(case, seed):
    """Conserved state of a perturbed Taylor-Green vortex: five float64
    tensors of shape (nz, ny, nx) on the GPU, one ideal gas with gamma 1.4."""
    n = _n(case)
    g = np.random.default_rng(seed)
    x, y, z = (torch.arange(m, dtype=torch.float64, device="cuda") * (TWO_PI / m) for m in n)
    X, Y, Z = x[None, None, :], y[None, :, None], z[:, None, None]
    a = g.uniform(0.95, 1.05)
    vel = [a * torch.sin(X) * torch.cos(Y) + 0 * Z, -a * torch.cos(X) * torch.sin(Y) + 0 * Z,
           torch.zeros(n[::-1], dtype=torch.float64, device="cuda")]
    for c in range(3):   # the solenoidal shear modes that break the symmetry
        ph = g.uniform(0, TWO_PI, 2)
        s, t = [(Y, Z), (X, Z), (X, Y)][c]
        vel[c] = vel[c] + 0.05 * g.standard_normal() * torch.sin(2 * s + ph[0]) * torch.cos(t + ph[1])
    p = 71.43 * g.uniform(0.9, 1.1)
    rho = torch.ones(n[::-1], dtype=torch.float64, device="cuda") * g.uniform(0.9, 1.1)
    ke = 0.5 * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)
    return [rho, rho * vel[0], rho * vel[1], rho * vel[2], p / 0.4 + rho * ke]


SCHEMES = {"c6": ch.lele_d1_6, "c10": ch.lele_d1_10, "c4": ch.pade_d1_4, "c8": ch.compact_filter}


def prepare(case, seed):
    ctx = ch.Context(0)
    kind = case["kind"]
    if kind in ("gradient", "filter"):
        n = _n(case)
        per = (case["periodic"],) * 3
        dt = np.float64 if case["dtype"] == "fp64" else np.float32
        decomp = ch.Decomp(n, per)
        plans = []
        for d in range(3):
            h = TWO_PI / (n[d] if case["periodic"] else n[d] - 1)
            plans.append(ch.plan_direction(ctx, decomp, SCHEMES[case["scheme"]](), d + 1, h, dtype=dt))
        f = ch.field(ctx, decomp, dt)
        view = _interior(f, decomp)
        view.copy_(_smooth_field(case, seed))
        state = dict(kind=kind, ctx=ctx, decomp=decomp, plans=plans, f=f, view=view)
        if kind == "gradient":
            state["out"] = [ch.field(ctx, decomp, dt) for _ in range(3)]
            state["views"] = [_interior(a, decomp) for a in state["out"]]
        torch.cuda.synchronize()
        return state
    if kind == "tgv":
        prob = ch.Problem(domain=((0.0, TWO_PI),) * 3, bcs=((ch.PeriodicBC(), ch.PeriodicBC()),) * 3,
                          ic=lambda X, Y, Z: None, name="taylor-green")
        num = ch.Numerics(n_global=_n(case), precision=case["dtype"], cfl=0.5)
        solver = ch.Solver(ctx, prob, num)
        Q = solver.allocate_state()
        sl = tuple(slice(solver.halo[d], solver.halo[d] + solver.n[d]) for d in range(3))
        for c, q in enumerate(_tgv_state(case, seed)):
            Q[sl + (c,)] = q.cpu().numpy().T
        solver.upload(Q)
        return dict(kind=kind, ctx=ctx, solver=solver, Q=Q, steps=case["steps"], single=False)
    # these programs keep what the mixed form computes as single-precision records
    single = case["dtype"] == "fp32"
    if kind == "shock":
        prob, num, Q = workloads.shock_problem(ch, (case["nx"], case["ny"], 1), case["dtype"])
        solver = ch.Solver(ctx, prob, num)
        # the seed's own interface: the composition is left as it is, and the
        # density and energy carry a small smooth disturbance along y
        g = np.random.default_rng(seed)
        hy = solver.halo[1]
        y = np.arange(case["ny"]) * (TWO_PI / case["ny"])
        fac = 1 + sum(0.01 * g.standard_normal() * np.cos(k * y + g.uniform(0, TWO_PI)) for k in (1, 2, 3))
        Q[:, hy:hy + case["ny"]] *= fac[None, :, None, None]
        solver.upload(Q)
        return dict(kind=kind, ctx=ctx, solver=solver, Q=Q, steps=case["steps"], single=single)
    # the lengths belong to the case, the driver pressures and densities to the seed
    specs = workloads.tube_specs(case["count"], seed=seed, nmin=case["nmin"], nmax=case["nmax"])
    lengths = np.random.default_rng(case["count"]).integers(case["nmin"], case["nmax"] + 1, case["count"])
    for spec, m in zip(specs, lengths):
        spec["n"] = int(m)
    batch = workloads.tube_batch(ctx, specs, precision=case["dtype"])
    return dict(kind=kind, ctx=ctx, batch=batch, steps=case["steps"], count=case["count"], single=single)


def run(state):
    kind = state["kind"]
    if kind == "gradient":
        for plan, out in zip(state["plans"], state["out"]):
            ch.apply_along_(out, plan, state["f"], state["decomp"])
        return state["views"]
    if kind == "filter":
        ch.filter_field_(state["f"], state["plans"], state["decomp"])
        return state["view"]
    if kind in ("tgv", "shock"):
        solver, Q = state["solver"], state["Q"]
        ch.run_(solver, Q, 1e9, nmax=solver.step_count + state["steps"])
        return Q.astype(np.float32) if state["single"] else Q
    batch = state["batch"]
    taken, dts = batch.run(max_steps=state["steps"], record=state["steps"])
    H = 4
    Q = np.concatenate([batch.download(i, H)[H:-H, 0, 0, :] for i in range(state["count"])])
    if state["single"]:
        Q, dts = Q.astype(np.float32), dts.astype(np.float32)
    return {"Q": Q, "dts": dts, "taken": taken}


def work(case):
    """Bytes and operations of one pass.  Operators read their field once and
    write each result once.  A step of run! cannot do without reading and
    writing the FP64 state and Runge-Kutta register in each of its five stages
    (the register is not read in the first) and the state once more for the
    filter; a pass also returns the state."""
    kind = case["kind"]
    if kind in ("gradient", "filter"):
        N = case["nx"] * case["ny"] * case["nz"]
        w = 8 if case["dtype"] == "fp64" else 4
        per = {"c4": 10, "c6": 14, "c10": 24, "c8": 22}[case["scheme"]]
        return {"bytes": w * N * (4 if kind == "gradient" else 2), "flops": 3 * per * N}
    if kind == "tubes":
        N, C, D, S = case["count"] * (case["nmin"] + case["nmax"]) / 2, 6, 1, 2
    elif kind == "shock":
        N, C, D, S = case["nx"] * case["ny"], 6, 2, 2
    else:
        N, C, D, S = case["nx"] * case["ny"] * case["nz"], 5, 3, 1
    state = 8.0 * C * N
    # line operators of one stage: gradients, divergences, sensor smoothing
    lines = D * (3 + 1 + (S if S > 1 else 0) + C) * 14 + D * (2 + (S if S > 1 else 0)) * 22
    stage = lines + 60 + 12 * D * (2 + S) + 30 * D * C
    return {"bytes": case["steps"] * (5 * 4 - 1 + 2) * state + state,
            "flops": N * case["steps"] * (5.0 * stage + 22 * D * C)}


# --------------------------------------------------------------------------
# The same results in 64-bit torch, from the schemes' definitions
# --------------------------------------------------------------------------
def _scheme_matrix(name, n, periodic, h):
    """Dense matrix of a compact scheme on n points: the left-hand band and the
    right-hand stencil row by row, solved together."""
    third = 1.0 / 3.0
    af = 0.45
    lhs, rhs, sym, a0 = {
        "c4": ([0.25], [0.75], False, 0.0),
        "c6": ([third], [7 / 9, 1 / 36], False, 0.0),
        "c10": ([0.5, 0.05], [17 / 24, 101 / 600, 1 / 600], False, 0.0),
        "c8": ([af], [(7 + 18 * af) / 32, (-7 + 14 * af) / 64, (1 - 2 * af) / 32, (-1 + 2 * af) / 256], True,
               (93 + 70 * af) / 128)}[name]
    A, B = np.eye(n), np.zeros((n, n))
    for i in range(n):
        for s, a in enumerate(lhs, 1):
            for j in (i - s, i + s):
                if periodic or 0 <= j < n:
                    A[i, j % n] += a
        B[i, i] += a0
        for m, c in enumerate(rhs, 1):
            for j, sg in ((i + m, 1.0), (i - m, 1.0 if sym else -1.0)):
                if periodic or 0 <= j < n:
                    B[i, j % n] += sg * c
    if not periodic:   # edge closures: (left-hand entries from the edge, right-hand weights)
        edge = [([1, 2], [-2.5, 2.0, 0.5]), ([0.25, 1, 0.25], [-0.75, 0.0, 0.75]),
                ([0, third, 1, third, 0], [-1 / 36, -7 / 9, 0.0, 7 / 9, 1 / 36])]
        for i, (left, right) in enumerate(edge[:{"c4": 1, "c6": 2, "c10": 3}[name]]):
            for k, sg in ((0, 1.0), (1, -1.0)):
                at = (lambda j: j) if k == 0 else (lambda j: n - 1 - j)
                A[at(i)], B[at(i)] = 0.0, 0.0
                for j, v in enumerate(left):
                    A[at(i), at(j)] = v
                for j, v in enumerate(right):
                    B[at(i), at(j)] = sg * v
    M = np.linalg.solve(A, B)
    return torch.from_numpy(M if sym else M / h).cuda()


def _along(M, f, axis):
    """M applied along x (0), y (1) or z (2) of a (nz, ny, nx) tensor."""
    if axis == 0:
        return torch.matmul(f, M.T.contiguous())
    if axis == 1:
        return torch.matmul(M, f)
    return torch.matmul(M, f.reshape(f.shape[0], -1)).reshape(f.shape)


LSRK_A = (0.0, -567301805773.0 / 1357537059087.0, -2404267990393.0 / 2016746695238.0,
          -3550918686646.0 / 2091501179385.0, -1275806237668.0 / 842570457699.0)
LSRK_B = (1432997174477.0 / 9575080441755.0, 5161836677717.0 / 13612068292357.0,
          1720146321549.0 / 2090206949498.0, 3134564353537.0 / 4481467310338.0,
          2277821191437.0 / 14882151754819.0)


def _tgv_exact(case, seed):
    """The periodic one-gas run in 64 bits: C6 derivatives, C8 filter, Cook
    artificial viscosities and conductivity, LSRK(5,4), cfl 0.5."""
    n = _n(case)
    h = [TWO_PI / m for m in n]
    D = [_scheme_matrix("c6", n[d], True, h[d]) for d in range(3)]
    F = [_scheme_matrix("c8", n[d], True, h[d]) for d in range(3)]
    Q = _tgv_state(case, seed)
    cv, R = 1.0 / 0.4, 1.0
    cp = cv + R
    mu = beta = kappa = torch.zeros_like(Q[0])

    def primitives():
        rho = Q[0]
        v = [Q[1 + i] / rho for i in range(3)]
        e = Q[4] / rho - 0.5 * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
        T = e / cv
        return rho, v, e, T, rho * R * T, torch.sqrt((1 + R / cv) * R * T)

    def smooth(f):
        for d in range(3):
            f = _along(F[d], f, d)
        return f

    def delta4(f, power):
        out = torch.zeros_like(f)
        for d in range(3):
            ax = 2 - d
            s = [torch.roll(f, -m, ax) for m in (-2, -1, 0, 1, 2)]
            out += h[d] ** power * (s[0] - 4 * s[1] + 6 * s[2] - 4 * s[3] + s[4]).abs()
        return out

    du = [torch.zeros_like(q) for q in Q]
    for _ in range(case["steps"]):
        rho, v, e, T, p, c = primitives()
        rate = sum((v[d].abs() + c) / h[d] for d in range(3))
        rate = rate + 2 * ((mu + beta) / rho + kappa / (rho * cp)) * sum(1 / x ** 2 for x in h)
        dt = 0.5 / float(rate.max())
        for A, B in zip(LSRK_A, LSRK_B):
            rho, v, e, T, p, c = primitives()
            G = [[_along(D[d], v[j], d) for j in range(3)] for d in range(3)]   # G[d][j] = d v_j / d x_d
            S2 = sum((0.5 * (G[a][b] + G[b][a])) ** 2 for a in range(3) for b in range(3))
            rs = rho * smooth(delta4(torch.sqrt(S2), 2)).clamp(min=0)
            mu, beta = 0.002 * rs, 1.0 * rs
            kappa = 0.01 * rho * c / T * smooth(delta4(e, 1)).clamp(min=0)
            div = G[0][0] + G[1][1] + G[2][2]
            dQ = [torch.zeros_like(q) for q in Q]
            for d in range(3):
                tau = [mu * (G[d][j] + G[j][d]) + ((beta - 2 / 3 * mu) * div if j == d else 0) for j in range(3)]
                flux = [rho * v[d]] + [rho * v[d] * v[j] + (p if j == d else 0) - tau[j] for j in range(3)]
                flux.append((Q[4] + p) * v[d] - sum(v[j] * tau[j] for j in range(3)) - kappa * _along(D[d], T, d))
                for i in range(5):
                    dQ[i] -= _along(D[d], flux[i], d)
            for i in range(5):
                du[i] = A * du[i] + dt * dQ[i]
                Q[i] = Q[i] + B * du[i]
        Q = [smooth(q) for q in Q]
    H = 4
    out = np.zeros(tuple(m + 2 * H for m in n) + (5,), order="F")
    for i in range(5):
        out[H:-H, H:-H, H:-H, i] = Q[i].cpu().numpy().T
    return out


def exact(case, seed):
    """run()'s answer in 64 bits.  The two-dimensional shock and the batches of
    tubes (hundreds of separate small problems) would take minutes this way."""
    if case["kind"] == "tgv":
        return _tgv_exact(case, seed)
    if case["kind"] not in ("gradient", "filter"):
        return None
    n = _n(case)
    f = _smooth_field(case, seed).to(_real(case)).double()
    M = [_scheme_matrix(case["scheme"], n[d], case["periodic"],
                        TWO_PI / (n[d] if case["periodic"] else n[d] - 1)) for d in range(3)]
    if case["kind"] == "gradient":
        return [_along(M[d], f, d) for d in range(3)]
    for d in range(3):
        f = _along(M[d], f, d)
    return f
