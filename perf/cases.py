"""The work a user of this framework has it do, as cases that can be timed.

Each case is one pass through a public entry point of `gputo` (or of the C
ABI behind it), on the sizes of this repository's configurations, tests and
benchmark, and on ragged ones between them:

  mgcg1    the MATLAB-facing solve on host arrays, `gputo.mgcg1`
  mgcg9    the CrossWalk/QNC solve on host arrays, `gputo.mgcg9`
  solve    `Solver.solve` on host arrays (FP64 or mixed precision)
  solve_d  `gputo_solve_d`: the same solve on device arrays
  design   a design run: `TopOpt`, a few design iterations, the state read back
  homog    `Solver.homogenize`: the elasticity tensor of a periodic cell
  matvec   `gputo_matvec_f64_noalloc`: the level-0 operator on device arrays
  grad     `Solver.learn_grad`: forward and backward of the learned stage's network

Solves run to a relative residual of 1e-10 (the tolerance of the 48x24x24
configuration), so a result is the solution of its problem to about ten
digits whatever path the iteration took.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-to_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import gputo  # noqa: E402

TOL = 1e-10
MAXIT = 500
EMIN = 1e-9
RMIN = math.sqrt(3.0)
# the benchmark's sweep schedule of the FP32 V-cycle: 1 + 3 on level 0, the
# prerelaxed iterate and 1 on level 1, 1 + 1 on level 2, 8 + 8 from level 3
SCHEDULE = dict(mixed_npre0=1, mixed_npost0=3, mixed_npre1=-1, mixed_npost1=1, mixed_npre2=1, mixed_npost2=1,
                mixed_npre3=8, mixed_npost3=8)
# the six layers of the level-2 network: channels in, channels out, stride
NET = [(4, 16, 1), (16, 32, 2), (32, 64, 2), (64, 32, 1), (32, 16, 1), (16, 3, 1)]


def _mesh(kind, nelx, nely, nelz, nl, **more):
    return dict(kind=kind, nelx=nelx, nely=nely, nelz=nelz, nl=nl, **more)


def listed():
    return [
        # the smallest call: a first try of the MEX on a coarse mesh, all latency
        dict(_mesh("mgcg1", 16, 8, 8, 3, density="start"), name="mgcg1_16x8x8"),
        # the everyday MEX call of the Cantilever drivers, mid-design density
        dict(_mesh("mgcg1", 48, 24, 24, 4, density="smooth"), name="mgcg1_48x24x24"),
        # the CrossWalk/QNC engine on a mesh that is no power of two in any direction
        dict(_mesh("mgcg9", 44, 28, 36, 3, density="smooth", nswp=2), name="mgcg9_44x28x36"),
        # a mixed-precision solve inside a device-resident program, medium mesh, default sweeps
        dict(_mesh("solve_d", 96, 48, 48, 4, density="smooth", precision=1, schedule="preset"),
             name="solve_d_mixed_96x48x48"),
        # the reference arithmetic at the benchmark's size, device-resident
        dict(_mesh("solve_d", 192, 96, 96, 5, density="start", precision=0, schedule="preset"),
             name="solve_d_f64_192x96x96"),
        # the benchmark's mixed solve called with host arrays, as the MEX does
        dict(_mesh("solve", 192, 96, 96, 5, density="start", precision=2, schedule="bench"),
             name="solve_mixed_192x96x96"),
        # the MATLAB preset's design loop on its 48x24x24 configuration
        dict(_mesh("design", 48, 24, 24, 4, preset=1, precision=0, schedule="preset", ft=1, iters=5),
             name="design_cfg0_48x24x24"),
        # a design run with the volume-preserving projection, FP64, ragged mesh
        dict(_mesh("design", 80, 40, 56, 4, preset=0, precision=0, schedule="preset", ft=3, iters=3),
             name="design_projected_80x40x56"),
        # the benchmark's design loop: restart a design, some iterations, read the state
        dict(_mesh("design", 192, 96, 96, 5, preset=0, precision=2, schedule="bench", ft=1, iters=4),
             name="design_mixed_192x96x96"),
        # periodic homogenisation of an inclusion cell, six load cases together
        dict(_mesh("homog", 48, 48, 48, 4, precision=0), name="homog_48x48x48"),
        # the operator alone in a serving loop: the largest mesh, nothing allocated
        dict(_mesh("matvec", 192, 96, 96, 5), name="matvec_192x96x96"),
        # training the learned stage: loss gradient of its network on the level-2 grid
        dict(_mesh("grad", 192, 96, 96, 5), name="learn_grad_192x96x96"),
    ]


def draw(rng):
    kind = rng.choice(["mgcg1", "mgcg1", "mgcg9", "solve", "solve_d", "solve_d", "design", "design", "homog", "matvec",
                       "grad"])
    for _ in range(1000):
        nl = rng.choice([4, 5]) if kind == "grad" else rng.choice([3, 3, 4, 4, 5])
        f = 1 << (nl - 1)
        c = (rng.randint(3, 12), rng.randint(2, 7), rng.randint(2, 7))
        if kind == "homog":
            c = (rng.randint(2, 6), rng.randint(2, 6), rng.randint(2, 6))
        size = [f * v for v in c]
        if size[0] * size[1] * size[2] <= (250_000 if kind == "homog" else 1_200_000):
            break
    if kind == "matvec":  # any mesh: the operator knows no levels
        size = [rng.randint(v, v + f) for v in size]
    case = _mesh(kind, *size, nl)
    precision = rng.choice([0, 1, 2])
    schedule = "bench" if precision and nl >= 4 and rng.random() < 0.5 else "preset"
    density = rng.choice(["start", "smooth"])
    if kind == "mgcg1":
        case.update(density=density)
    elif kind == "mgcg9":
        case.update(density=density, nswp=rng.choice([1, 2, 3]))
    elif kind in ("solve", "solve_d"):
        case.update(density=density, precision=precision, schedule=schedule)
    elif kind == "design":
        preset = rng.choice([0, 0, 1]) if precision == 0 else 0
        case.update(preset=preset, precision=precision, schedule=schedule, ft=rng.choice([1, 3]),
                    iters=rng.randint(1, 3))
    elif kind == "homog":
        case.update(precision=rng.choice([0, 1]))
    return case


# ---- inputs ------------------------------------------------------------------

def _sizes(case):
    return case["nelx"], case["nely"], case["nelz"]


def _counts(case):
    nx, ny, nz = _sizes(case)
    return nx * ny * nz, 3 * (nx + 1) * (ny + 1) * (nz + 1)


def _box3(a):
    """Mean over 3x3x3 neighbours (faces repeated)."""
    for ax in range(3):
        p = np.take(a, np.clip(np.arange(-1, a.shape[ax] + 1), 0, a.shape[ax] - 1), axis=ax)
        n = a.shape[ax]
        a = (np.take(p, np.arange(n), axis=ax) + np.take(p, np.arange(1, n + 1), axis=ax)
             + np.take(p, np.arange(2, n + 2), axis=ax)) / 3.0
    return a


def _density(case, seed):
    """Element densities: "start" is a design loop's first field (0.12 with a
    small perturbation), "smooth" a filtered field over [0.05, 1]."""
    nx, ny, nz = _sizes(case)
    rng = np.random.default_rng(seed)
    if case.get("density", "start") == "start":
        return 0.12 + rng.uniform(-0.01, 0.01, nx * ny * nz)
    r = _box3(rng.uniform(size=(nx, nz, ny)))
    return (0.05 + 0.95 * (r - r.min()) / (r.max() - r.min())).ravel()


def _cell(case, seed):
    """A periodic cell: a smooth wrapped field around 0.3 with a soft spherical inclusion."""
    nx, ny, nz = _sizes(case)
    x = np.random.default_rng(seed).uniform(size=(nx, nz, ny))
    for ax in range(3):
        x = (np.roll(x, 1, ax) + x + np.roll(x, -1, ax)) / 3.0
    x = np.clip(x - x.mean() + 0.3, 0.02, 1.0)
    g = np.meshgrid(*[(np.arange(n) + 0.5) / n - 0.5 for n in (nx, nz, ny)], indexing="ij")
    x[sum(v * v for v in g) <= 0.0625] = 0.1
    return x.ravel()


def _simp(x):
    return EMIN + x ** 3 * (1.0 - EMIN)


def _net_params(seed):
    rng = np.random.default_rng(seed)
    parts = []
    for ci, co, _ in NET:
        parts += [rng.normal(0.0, math.sqrt(2.0 / (27 * ci)), co * ci * 27), rng.normal(0.0, 0.02, co)]
    return np.concatenate(parts).astype(np.float32).astype(np.float64)


def _net_io(case, seed):
    nx, ny, nz = (v // 4 + 1 for v in _sizes(case))
    rng = np.random.default_rng(seed + 7)
    x = rng.normal(size=(4, nx, nz, ny))
    x[3] = 0.3 + 0.5 * rng.uniform(size=x[3].shape)  # the stiffness channel
    gy = rng.normal(size=(3, nx, nz, ny))
    return [v.astype(np.float32).astype(np.float64) for v in (x, gy)]


def _solver(case, **more):
    kw = dict(SCHEDULE) if case.get("schedule") == "bench" else {}
    if case.get("precision") == 2 and case.get("schedule") == "bench":
        kw["l0_kernel"] = 3  # split-BF16 MFMA (hi + lo), as the benchmark
    return gputo.Solver(*_sizes(case), case["nl"], preset=case.get("preset", 0), precision=case.get("precision", 0),
                        **kw, **more)


def prepare(case, seed):
    kind = case["kind"]
    nx, ny, nz = _sizes(case)
    Ke, F, fixed = gputo.cantilever(nx, ny, nz)
    st = dict(case=case, Ke=Ke, F=F, fixed=fixed)
    if kind in ("mgcg1", "mgcg9", "solve", "solve_d"):
        st["CX"] = _simp(_density(case, seed))
    if kind in ("mgcg1", "mgcg9"):
        st["U"] = np.zeros(F.size)
    elif kind == "solve":
        st["solver"] = _solver(case)
        st["U"] = np.zeros(F.size)
    elif kind == "solve_d":
        st["solver"] = _solver(case)
        st["d"] = [torch.from_numpy(v).cuda() for v in (F, st["CX"], (fixed - 1).astype(np.int32))]
        st["dU"] = torch.zeros(F.size, dtype=torch.float64, device="cuda")
    elif kind == "design":
        st["solver"] = _solver(case)
        st["x0"] = _density(case, seed)
        st["cfg"] = dict(volfrac=0.12, penal=3.0, rmin=RMIN, eta=0.4, beta=2.0, move=0.2, Emin=EMIN, E0=1.0,
                         ft=case["ft"], cg_tol=TOL, cg_maxit=MAXIT)
    elif kind == "homog":
        st["solver"] = _solver(case, periodic=True)
        st["CX"] = _simp(_cell(case, seed))
    elif kind == "matvec":
        rng = np.random.default_rng(seed)
        st["lib"] = gputo.load()
        u = rng.uniform(-1.0, 1.0, F.size)
        st["d"] = [torch.from_numpy(v).cuda() for v in (_simp(_density(case, seed)), u, (fixed - 1).astype(np.int32))]
        st["y"] = torch.zeros(F.size, dtype=torch.float64, device="cuda")
    elif kind == "grad":
        st["solver"] = gputo.Solver(nx, ny, nz, case["nl"], precision=gputo.PREC_MIXED_F32, learned=True)
        st["solver"].learn_params(_net_params(seed))
        st["x"], st["gy"] = _net_io(case, seed)
    else:
        raise ValueError(kind)
    return st


def _done(rc, what):
    if rc != 0:
        raise RuntimeError("%s: %s" % (what, rc))


def _addr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    Ke, F, fixed = state["Ke"], state["F"], state["fixed"]
    nx, ny, nz = _sizes(case)
    nl = case["nl"]
    if kind == "mgcg1":
        relres, nit = gputo.mgcg1(Ke, F, state["U"], state["CX"], fixed, len(fixed), nx, ny, nz, nl, TOL, MAXIT)
        _done(min(nit, 0), "mgcg1")
        return state["U"]
    if kind == "mgcg9":
        relres, nit = gputo.mgcg9(Ke, F, state["U"], state["CX"], fixed, len(fixed), nx, ny, nz, nl, TOL, MAXIT,
                                  case["nswp"], 0, 0.3, 1.0, 1.0, 1.0)
        _done(min(nit, 0), "mgcg9")
        return state["U"]
    if kind == "solve":
        U, relres, nit, rc = state["solver"].solve(Ke, F, state["CX"], fixed, TOL, MAXIT, U=state["U"])
        _done(rc, "solve")
        return U
    if kind == "solve_d":
        s = state["solver"]
        dF, dCX, dfix = state["d"]
        relres, nit = ctypes.c_double(), ctypes.c_int()
        _done(s.lib.gputo_solve_d(s.h, Ke.ctypes.data_as(ctypes.c_void_p), _addr(dF), _addr(state["dU"]), _addr(dCX),
                                  _addr(dfix), len(fixed), TOL, MAXIT, ctypes.byref(relres), ctypes.byref(nit)),
              "gputo_solve_d")
        return state["dU"]
    if kind == "design":
        loop = gputo.TopOpt(state["solver"], Ke, state["x0"], F, fixed, **state["cfg"])
        for _ in range(case["iters"]):
            loop.iterate()
        out = loop.state()
        loop.close()
        return dict(x=out[0], xPhys=out[1], U=out[2])
    if kind == "homog":
        CH, relres, nit, _ = state["solver"].homogenize(Ke, state["CX"], TOL, MAXIT)
        return CH
    if kind == "matvec":
        dCX, du, dfix = state["d"]
        _done(state["lib"].gputo_matvec_f64_noalloc(nx, ny, nz, Ke.ctypes.data_as(ctypes.c_void_p), _addr(dCX),
                                                    _addr(du), _addr(dfix), len(fixed), _addr(state["y"]),
                                                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
              "gputo_matvec_f64_noalloc")
        return state["y"]
    g = state["solver"].learn_grad(state["x"], state["gy"])
    return g.astype(np.float32)  # FP32 numbers, which the entry point hands over widened


def work(case):
    """Inputs read and outputs written once; one operator application (24 x 24
    multiply-adds per element) for each equation system that is solved."""
    nel, ndof = _counts(case)
    kind = case["kind"]
    if kind == "grad":
        sizes = [nel // 64, nel // 512, nel // 4096, nel // 4096, nel // 512, nel // 64]
        macs = sum(27 * ci * co * n for (ci, co, _), n in zip(NET, sizes))
        return {"bytes": 8.0 * 7 * sizes[0] + 4.0 * 2 * 141427, "flops": 6.0 * macs}
    systems = {"design": case.get("iters", 1), "homog": 6}.get(kind, 1)
    if kind == "design":
        return {"bytes": 8.0 * (2 * ndof + 3 * nel), "flops": 1152.0 * nel * systems}
    if kind == "homog":
        return {"bytes": 8.0 * nel, "flops": 1152.0 * nel * systems}
    return {"bytes": 8.0 * (2 * ndof + nel), "flops": 1152.0 * nel}


# ---- the same results in 64 bits, without the framework ----------------------

_IE, _JE, _KE = (0, 1, 1, 0, 0, 1, 1, 0), (0, 0, 1, 1, 0, 0, 1, 1), (0, 0, 0, 0, 1, 1, 1, 1)


def _ke():
    """24x24 stiffness of the unit trilinear hex (E = 1, nu = 0.3), 2x2x2 Gauss points."""
    nu, g = 0.3, 1.0 / math.sqrt(3.0)
    c = 1.0 / ((1 + nu) * (1 - 2 * nu))
    D = np.zeros((6, 6))
    D[:3, :3] = c * nu
    D[range(3), range(3)] = c * (1 - nu)
    D[range(3, 6), range(3, 6)] = c * (1 - 2 * nu) / 2
    K = np.zeros((24, 24))
    for p in range(8):
        s, e, t = (g if p >> b & 1 else -g for b in range(3))
        B = np.zeros((6, 24))
        for a in range(8):
            sx, sy, sz = 2 * _IE[a] - 1, 2 * _JE[a] - 1, 2 * _KE[a] - 1
            d = (0.25 * sx * (1 + sy * e) * (1 + sz * t), 0.25 * sy * (1 + sx * s) * (1 + sz * t),
                 0.25 * sz * (1 + sx * s) * (1 + sy * e))
            for row, (i, j) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (2, 0))):
                B[row, 3 * a + i] += d[j]
                if i != j:
                    B[row, 3 * a + j] += d[i]
        K += B.T @ D @ B / 8.0
    return K


class _Elastic:
    """K(CX) on node grids [nx+1, nz+1, ny+1, 3] (periodic: [nx, nz, ny, 3]) in torch, 64 bits."""

    def __init__(self, case, CX, periodic=False):
        self.n = (case["nelx"], case["nelz"], case["nely"])
        self.per = periodic
        self.Ke = torch.from_numpy(_ke()).cuda()
        self.CX = torch.as_tensor(CX, dtype=torch.float64, device="cuda").reshape(*self.n, 1)
        self.free = None
        if not periodic:
            self.free = torch.ones([v + 1 for v in self.n] + [3], dtype=torch.float64, device="cuda")
            self.free[0] = 0.0  # the x = 0 face is clamped

    def gather(self, u):
        a, b, c = self.n
        if self.per:
            return torch.cat([torch.roll(u, (-_IE[q], -_KE[q], -_JE[q]), (0, 1, 2)) for q in range(8)], -1)
        return torch.cat([u[_IE[q]:_IE[q] + a, _KE[q]:_KE[q] + b, _JE[q]:_JE[q] + c] for q in range(8)], -1)

    def scatter(self, f):
        a, b, c = self.n
        parts = f.split(3, -1)
        if self.per:
            return sum(torch.roll(p, (_IE[q], _KE[q], _JE[q]), (0, 1, 2)) for q, p in enumerate(parts))
        y = torch.zeros([v + 1 for v in self.n] + [3], dtype=torch.float64, device="cuda")
        for q, p in enumerate(parts):
            y[_IE[q]:_IE[q] + a, _KE[q]:_KE[q] + b, _JE[q]:_JE[q] + c] += p
        return y

    def mul(self, u):
        y = self.scatter((self.gather(u) @ self.Ke) * self.CX)
        return y if self.free is None else y * self.free

    def solve(self, f, tol=1e-13, most=8000):
        d = self.scatter(torch.diagonal(self.Ke).expand(*self.n, 24) * self.CX)
        if self.free is not None:
            f = f * self.free
            d = torch.where(self.free > 0, d, torch.ones_like(d))
        u, r = torch.zeros_like(f), f.clone()
        z = r / d
        p, rz, r0 = z.clone(), float((r * z).sum()), float(f.norm())
        for it in range(most):
            q = self.mul(p)
            al = rz / float((p * q).sum())
            u += al * p
            r -= al * q
            if it % 50 == 49:
                r = f - self.mul(u)
            if float(r.norm()) <= tol * r0:
                break
            z = r / d
            new = float((r * z).sum())
            p = z + (new / rz) * p
            rz = new
        return u


def _load(case):
    """Unit total downward load over the nodes (i = nelx, k = 0)."""
    nx, ny, nz = _sizes(case)
    F = torch.zeros(nx + 1, nz + 1, ny + 1, 3, dtype=torch.float64, device="cuda")
    F[nx, 0, :, 2] = -1.0 / (ny + 1)
    return F


def _exact_design(case, seed):
    n = (case["nelx"], case["nelz"], case["nely"])
    nel = n[0] * n[1] * n[2]
    vf, eta, beta, move, penal = 0.12, 0.4, 2.0, 0.2, 3.0
    x = torch.from_numpy(_density(case, seed)).cuda().reshape(n)
    h = torch.zeros(1, 1, 3, 3, 3, dtype=torch.float64, device="cuda")
    for a in range(3):
        for b in range(3):
            for c in range(3):
                h[0, 0, a, b, c] = max(0.0, RMIN - math.sqrt((a - 1) ** 2 + (b - 1) ** 2 + (c - 1) ** 2))

    def filt(v):
        p = torch.nn.functional.pad(v[None, None], (1, 1, 1, 1, 1, 1), mode="replicate")[0, 0]
        return sum(h[0, 0, a, b, c] * p[a:a + n[0], b:b + n[1], c:c + n[2]]
                   for a in range(3) for b in range(3) for c in range(3))

    Hs = filt(torch.ones_like(x))
    F = _load(case)
    for _ in range(case["iters"]):
        xt = filt(x) / Hs
        dHs, xp = Hs, xt
        if case["ft"] == 3:
            def prj(e):
                return (math.tanh(beta * e) + torch.tanh(beta * (xt - e))) / (math.tanh(beta * e) + math.tanh(beta * (1 - e)))

            for _ in range(100):
                f = float(prj(eta).mean()) - vf
                if abs(f) <= 1e-6:
                    break
                se = 1.0 / torch.cosh(beta * (xt - eta))
                df = -beta / math.sinh(beta) * se * se * torch.sinh(xt * beta) * torch.sinh((1 - xt) * beta)
                eta -= f / float(df.mean())
            t = torch.tanh(beta * (xt - eta))
            dHs = Hs / (beta * (1 - t * t) / (math.tanh(beta * eta) + math.tanh(beta * (1 - eta))))
            xp = prj(eta)
        K = _Elastic(case, EMIN + xp ** penal * (1 - EMIN))
        U = K.solve(F)
        ue = K.gather(U)
        ce = ((ue @ K.Ke) * ue).sum(-1)
        dc = filt(-penal * (1 - EMIN) * xp ** (penal - 1) * ce / dHs)
        dv = filt((1.0 / nel / vf) / dHs)
        oc = x * torch.sqrt(-dc / dv)
        l1, l2 = 0.0, float(oc.sum()) / nel / vf
        while (l2 - l1) / (l2 + l1) > 1e-4:
            mid = 0.5 * (l1 + l2)
            new = torch.clamp(torch.maximum(torch.minimum(torch.minimum(oc / mid, x + move), torch.ones_like(x)),
                                            x - move), min=0.0)
            if float(new.mean()) > vf:
                l1 = mid
            else:
                l2 = mid
        x = new
    return dict(x=x.reshape(-1), xPhys=xp.reshape(-1), U=U.reshape(-1))


def _exact_homog(case, seed):
    K = _Elastic(case, _simp(_cell(case, seed)), periodic=True)
    lo = np.array([_IE, _JE, _KE], dtype=np.float64)  # local coordinates of the 8 nodes
    u0 = np.zeros((6, 24))
    for a in range(8):
        X, Y, Z = lo[:, a]
        for q, v in enumerate(((X, 0, 0), (0, Y, 0), (0, 0, Z), (Y / 2, X / 2, 0), (0, Z / 2, Y / 2),
                               (Z / 2, 0, X / 2))):
            u0[q, 3 * a:3 * a + 3] = v
    u0 = torch.from_numpy(u0).cuda()
    e = []
    for q in range(6):
        f = K.scatter((u0[q] @ K.Ke) * K.CX)
        e.append(u0[q] - K.gather(K.solve(f, 1e-12, 2500)))
    CH = torch.zeros(6, 6, dtype=torch.float64)
    for a in range(6):
        ka = (e[a] @ K.Ke) * K.CX
        for b in range(6):
            CH[a, b] = float((ka * e[b]).sum()) / K.CX.numel()
    return CH


def _exact_grad(case, seed):
    flat, (x, gy) = _net_params(seed), _net_io(case, seed)
    F = torch.nn.functional
    ps, o = [], 0
    for ci, co, _ in NET:
        for shape in ((co, ci, 3, 3, 3), (co,)):
            k = int(np.prod(shape))
            ps.append(torch.from_numpy(flat[o:o + k].reshape(shape)).requires_grad_())
            o += k

    def up(v, like):
        for ax in (2, 3, 4):
            v = v.repeat_interleave(2, ax)
        return v[:, :, :like.shape[2], :like.shape[3], :like.shape[4]]

    def conv(k, v):
        return F.conv3d(v, ps[2 * k], ps[2 * k + 1], stride=NET[k][2], padding=1)

    e1 = F.relu(conv(0, torch.from_numpy(x)[None]))
    e2 = F.relu(conv(1, e1))
    e3 = F.relu(conv(2, e2))
    a2 = F.relu(conv(3, e3))
    a1 = F.relu(conv(4, up(a2, e2) + e2))
    y = conv(5, up(a1, e1) + e1)
    (y * torch.from_numpy(gy)[None]).sum().backward()
    return torch.cat([p.grad.reshape(-1) for p in ps])


def exact(case, seed):
    kind = case["kind"]
    nel, _ = _counts(case)
    if kind == "grad":
        return _exact_grad(case, seed)
    if kind == "matvec":
        nx, ny, nz = _sizes(case)
        u = torch.from_numpy(np.random.default_rng(seed).uniform(-1.0, 1.0, _counts(case)[1])).cuda()
        K = _Elastic(case, _simp(_density(case, seed)))
        return K.mul(u.reshape(nx + 1, nz + 1, ny + 1, 3)).reshape(-1)
    if kind == "homog":
        return _exact_homog(case, seed) if nel <= 120_000 else None
    if nel * case.get("iters", 1) > 300_000:  # plain CG would take too long
        return None
    if kind == "design":
        return _exact_design(case, seed)
    U = _Elastic(case, _simp(_density(case, seed))).solve(_load(case)).reshape(-1)
    if kind in ("mgcg1", "mgcg9", "solve"):
        U[1::3] *= -1.0  # the MATLAB frame
    return U
