"""The work that users of duct_amd have it do, as cases that can be timed and compared.

Four kinds of call, each through the package's public entry points:

  solve    duct_amd.helm3d_batch, or helm3d_mixed_batch where `scheme` is set: the cross-plane
           Helmholtz / Poisson solves of a batch of Fourier-space fields.  `bounds` holds one
           character per field ('d': velocity, 'n': pressure), `fold` is the argument of set_fold.
  step     duct_amd.step.rk3_step: one full Runge-Kutta time step of u, v, w and p, in place.
  adjoint  duct_amd.adjoint.projection_step_autograd: one projection step forward and its
           gradient with respect to the three right-hand sides.
  wall     duct_amd.temperature.helm3d_temp: the mixed-boundary solve of a scalar (temperature).

Fields are complex128 (modes, m, m) [mode, z, y] on the device, the reference's (my, mz, 0:mx1).
"""
import functools
import math

import numpy as np
import torch

import duct_amd
from duct_amd import adjoint, solver, step, temperature

DEV = "cuda"
ALP = 1.0            # Lx = 2 pi
HELMHOLTZ = 1000.0   # alambda of the Dirichlet fields (1 / (beta nu dt) of a substep)
NU = 0.01
PROJ_C = 0.5         # (alpha + beta) dt of the projection step


def listed():
    return [
        # One velocity component on the smallest grid: a latency-bound call (tests, tutorials, the
        # per-field loops of a caller that does not batch).
        {"name": "solve_33x16_d", "kind": "solve", "m": 33, "modes": 16, "bounds": "d", "fold": 0, "scheme": ""},
        # u, v, w and p of one substep on the mid-size grid, the library's default arithmetic.
        {"name": "solve_129x64_dddn", "kind": "solve", "m": 129, "modes": 64, "bounds": "dddn", "fold": 0, "scheme": ""},
        # The same on a grid between the powers of two, with an even number of points.
        {"name": "solve_200x96_dddn", "kind": "solve", "m": 200, "modes": 96, "bounds": "dddn", "fold": 0, "scheme": ""},
        # The benchmark's workload: default, folded, and refined from half precision.
        {"name": "solve_257x256_dddn", "kind": "solve", "m": 257, "modes": 256, "bounds": "dddn", "fold": 0, "scheme": ""},
        {"name": "fold_257x256_dddn", "kind": "solve", "m": 257, "modes": 256, "bounds": "dddn", "fold": 2, "scheme": ""},
        {"name": "refine_257x256_dddn", "kind": "solve", "m": 257, "modes": 256, "bounds": "dddn", "fold": 0,
         "scheme": "fold16q"},
        # Whole time steps of the simulation: a small run (launch-bound), the mid-size production
        # grid, a ragged one whose x grid is not a multiple of 16, and a large one.
        {"name": "step_33x16", "kind": "step", "m": 33, "modes": 16, "mgalx": 48},
        {"name": "step_97x40", "kind": "step", "m": 97, "modes": 40, "mgalx": 120},
        {"name": "step_129x64", "kind": "step", "m": 129, "modes": 64, "mgalx": 192},
        {"name": "step_257x128", "kind": "step", "m": 257, "modes": 128, "mgalx": 384},
        # Gradients of flow functionals: forward projection step and backward.
        {"name": "adjoint_129x64", "kind": "adjoint", "m": 129, "modes": 64},
        # The temperature equation's solve on a rectangular grid, two walls of each type.
        {"name": "wall_97x129x64", "kind": "wall", "m": 97, "mz": 129, "modes": 64, "walls": "dndn"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth_even(x):
    """The smallest even x' >= x whose prime factors are 2, 3 and 5, as x grids are chosen for the FFT."""
    x += x % 2
    while True:
        r = x
        for p in (2, 3, 5):
            while r % p == 0:
                r //= p
        if r == 1:
            return x
        x += 2


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "step", "step", "step", "adjoint", "wall"])
    if kind == "solve":
        how = rng.choice(["default", "default", "fold", "refine"])
        # the folded bases start at 65 interior points
        m = _log_int(rng, 17 if how == "default" else 67, 257)
        modes = _log_int(rng, 4, 256)
        bounds = rng.choice(["d", "n", "ddd", "dddn"])
        return {"kind": kind, "m": m, "modes": modes, "bounds": bounds, "fold": 2 if how == "fold" else 0,
                "scheme": "fold16q" if how == "refine" else ""}
    if kind == "step":
        m, modes = _log_int(rng, 17, 257), _log_int(rng, 4, 128)
        return {"kind": kind, "m": m, "modes": modes, "mgalx": _smooth_even(3 * modes)}
    m, modes = _log_int(rng, 17, 161), _log_int(rng, 4, 96)
    if kind == "adjoint":
        return {"kind": kind, "m": m, "modes": modes}
    return {"kind": kind, "m": m, "mz": _log_int(rng, 17, 161), "modes": modes,
            "walls": "".join(rng.choice("dn") for _ in range(3)) + "d"}


# ---- inputs ----------------------------------------------------------------------------------

_grid = {"m": None, "wall": None}


def _setup(m):
    """The eigenbases of the m-point grid, set up once as a program does that stays on its grid."""
    if _grid["m"] != m:
        duct_amd.init(torch.cuda.current_device())
        duct_amd.setup(m)
        _grid["m"] = m


@functools.lru_cache(maxsize=8)
def _cheb(m, K):
    """T_p and T_p' at the nodes x_j = -cos(pi j / (m-1)), p < K, on the device: [node, p]."""
    C = np.polynomial.chebyshev
    x = -np.cos(np.pi * np.arange(m) / (m - 1))
    T = C.chebvander(x, K - 1)
    dT = np.stack([C.chebval(x, C.chebder(np.eye(K)[p])) for p in range(K)], axis=1)
    return torch.from_numpy(T).to(DEV), torch.from_numpy(dT).to(DEV), torch.from_numpy(x).to(DEV)


def _series(gen, modes, K, mode_decay):
    """Complex Chebyshev coefficients (modes, K, K) [mode, z, y] that decay with the degree."""
    a = torch.complex(torch.randn((modes, K, K), generator=gen, dtype=torch.float64, device=DEV),
                      torch.randn((modes, K, K), generator=gen, dtype=torch.float64, device=DEV))
    q = torch.arange(K, dtype=torch.float64, device=DEV)
    a = a * torch.exp(-0.15 * (q[:, None] + q[None, :]))
    a = a * torch.exp(-mode_decay * torch.arange(modes, dtype=torch.float64, device=DEV))[:, None, None]
    a[0] = torch.complex(a[0].real, torch.zeros_like(a[0].real))
    return a


def _nodal(Tz, a, Ty):
    """sum_qp Tz[l, q] a[k, q, p] Ty[j, p], real and imaginary parts apart."""
    f = [torch.matmul(torch.matmul(Tz, part.contiguous()), Ty.T.contiguous()) for part in (a.real, a.imag)]
    return torch.complex(f[0], f[1])


def _smooth_field(gen, m, mz, modes, zero_walls):
    K = min(m, mz, 64)
    f = _nodal(_cheb(mz, K)[0], _series(gen, modes, K, 0.0), _cheb(m, K)[0])
    if zero_walls:
        f[:, 0, :] = 0
        f[:, -1, :] = 0
        f[:, :, 0] = 0
        f[:, :, -1] = 0
    return f


def _velocity(gen, m, modes):
    """A laminar-like mean flow plus 5% of a divergence-free perturbation that vanishes on the walls."""
    K = min(24, m - 5)
    T, dT, x = _cheb(m, K)
    g, dg = (1 - x * x) ** 2, -4.0 * x * (1 - x * x)
    gz, gy, dgz, dgy = g[:, None], g[None, :], dg[:, None], dg[None, :]
    A, Ay, Az = [], [], []
    for _ in range(3):
        a = _series(gen, modes, K, 0.2)
        h, hy, hz = _nodal(T, a, T), _nodal(T, a, dT), _nodal(dT, a, T)
        A.append(gz * gy * h)
        Ay.append(gz * (dgy * h + gy * hy))
        Az.append(gy * (dgz * h + gz * hz))
    ik = 1j * ALP * torch.arange(modes, dtype=torch.float64, device=DEV)[:, None, None]
    vel = [Ay[2] - Az[1], Az[0] - ik * A[2], ik * A[1] - Ay[0]]
    scale = 0.05 / max(float(f.abs().max()) for f in vel)
    vel = [(scale * f).contiguous() for f in vel]
    vel[0][0] += (1 - x * x)[:, None] * (1 - x * x)[None, :]
    return vel


def _dt(case):
    return 0.5 / case["modes"]   # an advective step below the scheme's limit at the finest wave


def _inputs(case, seed):
    """The seeded input fields of one case, in a fixed order."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) * 7919 + 17)
    m, modes = case["m"], case["modes"]
    if case["kind"] == "solve":
        return [_smooth_field(gen, m, m, modes, b == "d") for b in case["bounds"]]
    if case["kind"] == "step":
        vel = _velocity(gen, m, modes)
        return vel + [torch.zeros_like(vel[0]) for _ in range(4)]          # p and the three old advection terms
    if case["kind"] == "adjoint":
        return [_smooth_field(gen, m, m, modes, True) for _ in range(6)]    # fu, fv, fw and the output's gradients
    mz = case["mz"]
    walls = [0.1 * torch.randn((modes, 2, n), generator=gen, dtype=torch.float64, device=DEV) for n in (mz, m)]
    return [_smooth_field(gen, m, mz, modes, False)] + walls


def prepare(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    state = {"case": case}
    if kind == "wall":
        key = (case["m"], case["mz"], case["walls"])
        if _grid["wall"] != key:
            duct_amd.init(torch.cuda.current_device())
            temperature.setup_temp(case["m"], case["walls"], mz=case["mz"])
            _grid["wall"] = key
        state.update(rhs=x[0], bcy=x[1], bcz=x[2], sol=torch.empty_like(x[0]))
        return state
    _setup(case["m"])
    solver.set_fold(case.get("fold", 0))
    if kind == "solve":
        state.update(rhs=x, sol=[torch.zeros_like(f) for f in x],
                     alambda=[HELMHOLTZ if b == "d" else 0.0 for b in case["bounds"]])
    elif kind == "step":
        state.update(vel=x[:3], p=x[3], adv=x[4:], dt=_dt(case))
    else:
        state.update(f=[f.requires_grad_(True) for f in x[:3]], g=x[3:])
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "solve":
        args = (state["rhs"], state["sol"], case["bounds"], state["alambda"])
        if case["scheme"]:
            solver.helm3d_mixed_batch(*args, alp=ALP, scheme0=case["scheme"], scheme1=case["scheme"], niter=1)
        else:
            duct_amd.helm3d_batch(*args, alp=ALP)
        return state["sol"]
    if case["kind"] == "step":
        step.rk3_step(*state["vel"], state["p"], state["adv"], NU, state["dt"], case["mgalx"], alp=ALP)
        return state["vel"] + [state["p"]] + state["adv"]
    if case["kind"] == "adjoint":
        out = adjoint.projection_step_autograd(*state["f"], HELMHOLTZ, ALP, 0, PROJ_C)
        grad = torch.autograd.grad(out, state["f"], grad_outputs=state["g"])
        return [o.detach() for o in out] + list(grad)
    temperature.helm3d_temp(state["rhs"], state["sol"], state["bcy"], state["bcz"], HELMHOLTZ, alp=ALP)
    return state["sol"]


def work(case):
    """What a pass cannot do without: its inputs read and its outputs written once, and the
    multiplications of its eigenbasis products, derivative products and transforms.  The products
    of a reflection-symmetric basis (all but the mixed walls) take half of their dense count."""
    m, M = case["m"], case["modes"]
    n = m - 2
    if case["kind"] == "wall":
        nz = case["mz"] - 2
        dense = 2.0 * 2 * M * (2.0 * n * n * nz + 2.0 * n * nz * nz)   # four products of every real plane
        return {"bytes": 2.0 * 16 * m * case["mz"] * M + 16.0 * M * (m + case["mz"]), "flops": dense}
    field = 16.0 * m * m * M
    solve = 0.5 * 4 * 2.0 * n ** 3 * (2 * M - 1)
    deriv = 0.5 * 2.0 * m ** 3 * 2 * M
    if case["kind"] == "solve":
        nf = len(case["bounds"])
        return {"bytes": 2.0 * nf * field, "flops": nf * solve}
    if case["kind"] == "step":
        X = case["mgalx"]
        fft = 9 * 2.5 * X * math.log2(X) * m * m
        return {"bytes": 11.0 * field, "flops": 3.0 * (4 * solve + 20 * deriv + fft)}
    return {"bytes": 12.0 * field, "flops": 2.0 * (4 * solve + 4 * deriv)}


# ---- the same in plain 64-bit torch ------------------------------------------------------------

def _textbook(m):
    N = m - 1
    j = np.arange(m)
    x = -np.cos(np.pi * j / N)
    c = np.ones(m)
    c[0] = c[-1] = 2.0
    diff = x[:, None] - x[None, :]
    np.fill_diagonal(diff, 1.0)
    D = (c[:, None] / c[None, :]) * np.where((j[:, None] + j[None, :]) % 2, -1.0, 1.0) / diff
    i = np.arange(1, N)
    D[i, i] = -0.5 * x[i] / (1.0 - x[i] ** 2)
    D[0, 0] = -(2.0 * N * N + 1.0) / 6.0
    D[N, N] = -D[0, 0]
    return D


@functools.lru_cache(maxsize=2)
def _derivatives(m):
    """First and second collocation derivative matrices, formed in extended precision."""
    N = m - 1
    j = np.arange(m)
    pi = np.longdouble("3.14159265358979323846264338327950288")
    s = np.sin(pi * (j[:, None] + j[None, :]) / (2 * N)) * np.sin(pi * (j[:, None] - j[None, :]) / (2 * N)) * 2
    np.fill_diagonal(s, 1)                                    # x_i - x_k
    c = np.ones(m, dtype=np.longdouble)
    c[0] = c[-1] = 2
    D = (c[:, None] / c[None, :]) * np.where((j[:, None] + j[None, :]) % 2, -1, 1) / s
    np.fill_diagonal(D, 0)
    np.fill_diagonal(D, -D.sum(axis=1))
    return [torch.from_numpy(a.astype(np.float64)).to(DEV) for a in (D, D @ D)]


def _dev(*a):
    return [torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for v in a]


@functools.lru_cache(maxsize=2)
def _bases(m):
    """Per boundary type P, P^-1, the eigenvalues and what the Neumann walls need."""
    D = _textbook(m)
    D2, N, s = D @ D, m - 1, slice(1, m - 1)
    det = D[0, 0] * D[N, N] - D[0, N] * D[N, 0]
    c1 = D[0, N] * D[N, s] - D[N, N] * D[0, s]
    cm = D[N, 0] * D[0, s] - D[0, 0] * D[N, s]
    ops = {"d": np.ascontiguousarray(D2[s, s]),
           "n": np.ascontiguousarray(((D2[s, 0][:, None] * c1) / det + D2[s, s]) + (D2[s, N][:, None] * cm) / det)}
    out = {}
    for b, op in ops.items():
        lam, P = np.linalg.eig(op)
        lam, P = lam.real, P.real
        out[b] = _dev(P, np.linalg.inv(P), lam) + [int(np.argmin(np.abs(lam)))]
    AM = np.array([[2.0 * D[0, 0], D[0, N], 0.0, D[0, N]], [-D[N, 0], D[0, 0] - D[N, N], D[0, N], 0.0],
                   [0.0, D[N, 0], 2.0 * D[N, N], D[N, 0]], [-D[N, 0], 0.0, D[0, N], D[0, 0] - D[N, N]]])
    out["walls"] = _dev(D, np.linalg.inv(AM))
    return out


def _mul(A, f):
    """Real matrix times complex field along z: A f."""
    return torch.complex(torch.matmul(A, f.real.contiguous()), torch.matmul(A, f.imag.contiguous()))


def _lum(f, A):
    """Complex field times real matrix along y: f A."""
    return torch.complex(torch.matmul(f.real.contiguous(), A), torch.matmul(f.imag.contiguous(), A))


def _sandwich(A, f):
    return _lum(_mul(A, f), A.T.contiguous())


def _helm(f, bound, alambda):
    m, M = f.shape[-1], f.shape[0]
    P, Pi, lam, io = _bases(m)[bound]
    xl = alambda + (ALP * torch.arange(M, dtype=torch.float64, device=DEV)) ** 2
    den = lam[:, None] + lam[None, :] - xl[:, None, None]
    G = _sandwich(Pi, f[:, 1:-1, 1:-1])
    if bound == "n" and alambda == 0.0:     # the singular plane: u = 0 at the gauge node
        den = den.clone()
        den[0, io, io] = 1.0
        G = G / den
        keep = torch.ones_like(den)
        keep[0, io, io] = 0.0
        G = G * keep
        U = _sandwich(P, G)
        fix = torch.zeros_like(den)
        fix[0] = P[:, io][:, None] * P[:, io][None, :] / (P[io, io] * P[io, io])
        U = U - U[0, io, io] * fix
    else:
        U = _sandwich(P, G / den)
    U = torch.cat([torch.complex(U[:1].real, torch.zeros_like(U[:1].real)), U[1:]])   # Im is not solved at k = 0
    if bound == "d":
        return torch.view_as_complex(torch.nn.functional.pad(torch.view_as_real(U), (0, 0, 1, 1, 1, 1)).contiguous())
    D, AM1 = _bases(m)["walls"]
    D = D.to(torch.complex128)
    d0, dm = D[0, 1:-1], D[-1, 1:-1]
    det = D[0, 0] * D[-1, -1] - D[0, -1] * D[-1, 0]
    sb, st = torch.einsum("kzy,z->ky", U, d0), torch.einsum("kzy,z->ky", U, dm)
    sl, sr = torch.einsum("kzy,y->kz", U, d0), torch.einsum("kzy,y->kz", U, dm)
    vb, vt = (-D[-1, -1] * sb + D[0, -1] * st) / det, (D[-1, 0] * sb - D[0, 0] * st) / det
    el, er = (-D[-1, -1] * sl + D[0, -1] * sr) / det, (D[-1, 0] * sl - D[0, 0] * sr) / det
    ff = torch.stack([-(vb @ d0) - (el @ d0), (vb @ dm) - (er @ d0), -(vt @ dm) - (er @ dm), -(vt @ d0) + (el @ dm)], 1)
    cn = ff @ AM1.to(torch.complex128).T
    bottom = torch.cat([cn[:, 0:1], vb, cn[:, 1:2]], 1)[:, None, :]
    top = torch.cat([cn[:, 3:4], vt, cn[:, 2:3]], 1)[:, None, :]
    return torch.cat([bottom, torch.cat([el[:, :, None], U, er[:, :, None]], 2), top], 1)


def _dx(f, order=1):
    ik = 1j * ALP * torch.arange(f.shape[0], dtype=torch.float64, device=DEV)[:, None, None]
    return ik ** order * f


def _dy(f, D):
    return _lum(f, D.T.contiguous())


def _advection(u, v, w, X):
    M, m = u.shape[0], u.shape[-1]
    D = _derivatives(m)[0]

    def phys(f):
        full = torch.zeros((X // 2 + 1, m, m), dtype=torch.complex128, device=DEV)
        full[:M] = f
        return torch.fft.irfft(full, n=X, dim=0) * X

    def back(p):
        return torch.fft.rfft(p, dim=0)[:M] / X

    u, v, w = phys(u), phys(v), phys(w)
    uu, vv, ww, uv, uw, vw = (back(a * b) for a, b in ((u, u), (v, v), (w, w), (u, v), (u, w), (v, w)))
    return [_dx(uu) + _dy(uv, D) + _mul(D, uw), _dx(uv) + _dy(vv, D) + _mul(D, vw), _dx(uw) + _dy(vw, D) + _mul(D, ww)]


def _rk3(vel, p, adv, dt, X):
    m = p.shape[-1]
    D, D2 = _derivatives(m)
    ak, bk = (29 / 96, -3 / 40, 1 / 6), (37 / 160, 5 / 24, 1 / 6)
    gk, rk = (8 / 15, 5 / 12, 3 / 4), (0.0, -17 / 60, -5 / 12)
    dpdx = -NU * 3.39344926982230
    for a, b, g, r in zip(ak, bk, gk, rk):
        new = _advection(*vel, X)
        grad = [_dx(p), _dy(p, D), _mul(D, p)]
        h = []
        for c in range(3):
            lap = _dx(vel[c], 2) + _dy(vel[c], D2) + _mul(D2, vel[c])
            hc = -r * adv[c] - g * new[c] + NU * a * lap + vel[c] / dt - (a + b) * grad[c]
            if c == 0:
                hc[0] -= (a + b) * dpdx
            h.append(hc * (-1.0 / (NU * b)))
        adv = new
        vel = [_helm(hc, "d", 1.0 / (b * NU * dt)) for hc in h]
        phi = _helm((_dx(vel[0]) + _dy(vel[1], D) + _mul(D, vel[2])) / ((a + b) * dt), "n", 0.0)
        p = p + phi - (a + b) * dt * NU * (_dx(phi, 2) + _dy(phi, D2) + _mul(D2, phi))
        s = -dt * (a + b)
        vel = [vel[0] + s * _dx(phi), vel[1] + s * _dy(phi, D), vel[2] + s * _mul(D, phi)]
    return vel + [p] + adv


def _project(f):
    D = _derivatives(f[0].shape[-1])[0]
    us = [_helm(x, "d", HELMHOLTZ) for x in f]
    phi = _helm((_dx(us[0]) + _dy(us[1], D) + _mul(D, us[2])) / PROJ_C, "n", 0.0)
    return [us[0] - PROJ_C * _dx(phi), us[1] - PROJ_C * _dy(phi, D), us[2] - PROJ_C * _mul(D, phi)]


def _wall_line(D, t1, t2, v1, v2, a, b):
    """Values at both ends of a line from the wall data and the interior's shares a, b of the derivative rows."""
    if t1 == "d" and t2 == "d":
        return v1, v2
    if t1 == "d":
        return v1, (v2 - D[-1, 0] * v1 - b) / D[-1, -1]
    if t2 == "d":
        return (v1 - D[0, -1] * v2 - a) / D[0, 0], v2
    det = D[0, 0] * D[-1, -1] - D[0, -1] * D[-1, 0]
    return (D[-1, -1] * (v1 - a) - D[0, -1] * (v2 - b)) / det, (D[0, 0] * (v2 - b) - D[-1, 0] * (v1 - a)) / det


def _wall_basis(m, t1, t2):
    D = _textbook(m)
    D2, s, N = D @ D, slice(1, m - 1), m - 1
    op = D2[s, s].copy()
    if t1 == "n" and t2 == "n":
        det = D[0, 0] * D[N, N] - D[0, N] * D[N, 0]
        op = D2[s, :1] * (D[0, N] * D[N, s] - D[N, N] * D[0, s]) / det + op \
            + D2[s, N:] * (D[N, 0] * D[0, s] - D[0, 0] * D[N, s]) / det
    elif t2 == "n":
        op = op - D2[s, N:] * D[N, s] / D[N, N]
    elif t1 == "n":
        op = op - D2[s, :1] * D[0, s] / D[0, 0]
    E, P = np.linalg.eig(op)
    return _dev(D, D2, P.real, np.linalg.inv(P.real), E.real)


def _wall_solve(case, rhs, bcy, bcz):
    w = case["walls"]
    Dy, D2y, Py, Pyi, Ey = _wall_basis(case["m"], w[0], w[1])
    Dz, D2z, Pz, Pzi, Ez = _wall_basis(case["mz"], w[2], w[3])
    gy = _wall_line(Dy, w[0], w[1], bcy[:, 0, 1:-1], bcy[:, 1, 1:-1], 0.0, 0.0)
    gz = _wall_line(Dz, w[2], w[3], bcz[:, 0, 1:-1], bcz[:, 1, 1:-1], 0.0, 0.0)
    corr = sum(g[:, :, None] * D2y[1:-1, e][None, None, :] for g, e in zip(gy, (0, -1))) \
        + sum(D2z[1:-1, e][None, :, None] * g[:, None, :] for g, e in zip(gz, (0, -1)))
    F = rhs[:, 1:-1, 1:-1] - torch.complex(corr, corr)
    xl = HELMHOLTZ + (ALP * torch.arange(rhs.shape[0], dtype=torch.float64, device=DEV)) ** 2
    G = _lum(_mul(Pzi, F), Pyi.T.contiguous()) / (Ez[:, None] + Ey[None, :] - xl[:, None, None])
    U = rhs.clone()
    S = _lum(_mul(Pz, G), Py.T.contiguous())
    S[0] = torch.complex(S[0].real, torch.zeros_like(S[0].real))
    U[:, 1:-1, 1:-1] = S

    def both(v):
        return torch.complex(v, v)

    def share(row, sub):
        return torch.einsum(sub, S, row[1:-1].to(torch.complex128))

    e = _wall_line(Dy, w[0], w[1], both(bcy[:, 0, 1:-1]), both(bcy[:, 1, 1:-1]), share(Dy[0], "kzy,y->kz"),
                   share(Dy[-1], "kzy,y->kz"))
    U[:, 1:-1, 0], U[:, 1:-1, -1] = e
    e = _wall_line(Dz, w[2], w[3], both(bcz[:, 0, 1:-1]), both(bcz[:, 1, 1:-1]), share(Dz[0], "kzy,z->ky"),
                   share(Dz[-1], "kzy,z->ky"))
    U[:, 0, 1:-1], U[:, -1, 1:-1] = e
    U[0] = torch.complex(U[0].real, torch.zeros_like(U[0].real))
    return U


def exact(case, seed):
    x = _inputs(case, seed)
    if case["kind"] == "solve":
        return [_helm(f, b, HELMHOLTZ if b == "d" else 0.0) for f, b in zip(x, case["bounds"])]
    if case["kind"] == "step":
        return _rk3(x[:3], x[3], x[4:], _dt(case), case["mgalx"])
    if case["kind"] == "adjoint":
        f = [t.requires_grad_(True) for t in x[:3]]
        out = _project(f)
        return [o.detach() for o in out] + list(torch.autograd.grad(out, f, grad_outputs=x[3:]))
    return _wall_solve(case, *x)
