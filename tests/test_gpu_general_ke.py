"""The level-0 kernels that serve an element matrix without the isotropic modal
form: the node-gather in FP64 and FP32 (with the unit-H8 entry classes and
without) and the MFMA flavours, in every mode, in whole solves, in periodic cells
and in the matvec that allocates nothing.

Two matrices: "classes" scales each entry class of Ke0 by a factor of its own,
"full" adds a symmetric random matrix.  Operators take a perturbation of 1e-3,
solves one of 1e-9, which keeps them as well posed as with Ke0 and is far from
what passes as isotropic (1e-14).

Tolerances as with the isotropic Ke0: relative to max|y|, FP64 1e-13 (summation
order), FP32 2e-6, the hi+lo split 1e-4; solves to 1e-10 agree to 1e-7, mixed in
at most two iterations more than FP64 (the hi+lo split: 40); homogenised tensors
to 1e-8.  The FP64 solve follows the oracle's: its residual after ten iterations
agrees to 1e-6 of its value, the rounding of two summation orders times the growth
of as many iterations.  (The oracle's count is no function of the input: its
threads' sums are added in any order, and it ends this solve after 29 or 31
iterations, as 1e-10 falls.)"""
import ctypes
import os
import re

import numpy as np
import pytest

from conftest import ROOT, cantilever_case
from test_gpu_modal import references, rel
from test_zz_no_alloc import Dev

pytestmark = pytest.mark.gpu


def entry_classes():
    src = open(os.path.join(ROOT, "gpu-to_amd", "csrc", "ke_classes.h")).read()
    table = re.search(r"kKeClass\[576\] = \{([^}]*)\}", src).group(1)
    return np.array([int(v) for v in table.replace("\n", " ").split(",") if v.strip()]).reshape(24, 24)


def element(gputo, kind, size):
    Ke = gputo.ke0_h8()
    if kind == "classes":
        cls = entry_classes()
        first = [Ke[cls == k][0] for k in range(cls.max() + 1)]
        return np.ascontiguousarray(np.array(first)[cls] * (1.0 + size * (1.0 + cls)))
    E = np.random.default_rng(81).uniform(-1, 1, (24, 24)) * size
    return Ke + (E + E.T)


@pytest.mark.parametrize("kind", ["classes", "full"])
@pytest.mark.parametrize("mesh", [(16, 8, 8, 3), (40, 20, 12, 3)])
@pytest.mark.parametrize("kernel,tol", [(0, 1e-13), (1, 2e-6), (2, 2e-6), (3, 1e-4), (4, 2e-6)])
def test_level0_modes(gputo, oracle, kernel, tol, mesh, kind):
    """kernel 0: the FP64 node-gather."""
    nelx, nely, nelz, nl = mesh
    print("case", mesh, kernel, kind, flush=True)
    _, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=82, kind="smooth")
    Ke = element(gputo, kind, 1e-3)
    s = gputo.Solver(nelx, nely, nelz, nl, precision=2 if kernel else 0, l0_kernel=kernel)
    s.setup(Ke, CX, fixed)
    rng = np.random.default_rng(83)
    u, f = rng.uniform(-1, 1, F.size), rng.uniform(-1, 1, F.size)
    ad = oracle.prepad0(Ke, CX, nelx, nely, nelz)
    ref = references(lambda v: oracle.matvec0(Ke, CX, v, np.zeros(0), nelx, nely, nelz), u, f, ad,
                     (fixed - 1).astype(np.int64))
    for mode in range(5):
        y = s.level_apply(0, 1, mode, u, f, fp32=kernel > 0)
        assert rel(y, ref[mode]) < tol, (mode, rel(y, ref[mode]))
        assert np.array_equal(y, s.level_apply(0, 1, mode, u, f, fp32=kernel > 0))
    s.close()


@pytest.mark.parametrize("kind", ["classes", "full"])
@pytest.mark.parametrize("kw", [dict(), dict(preset=1), dict(preset=2, nswp=2), dict(precision=1, l0_kernel=1),
                                dict(precision=1, l0_kernel=2), dict(precision=2, l0_kernel=3),
                                dict(precision=2, l0_kernel=4), dict(precision=1, preset=2, nswp=2),
                                dict(precision=1, l0_kernel=1, graph_vcycles=1)])
def test_solve(gputo, oracle, kw, kind):
    nelx, nely, nelz, nl = 32, 16, 16, 4
    print("case", kw, kind, flush=True)
    _, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=84, kind="smooth")
    Ke = element(gputo, kind, 1e-9)
    preset = kw.get("preset", 0)
    Uo, _, no, rco = oracle.mgcg(Ke, F, CX, fixed, nelx, nely, nelz, nl, 1e-10, 300, preset=preset, nswp=2)
    s = gputo.Solver(nelx, nely, nelz, nl, **kw)
    U, r, n, rc = s.solve(Ke, F, CX, fixed, 1e-10, 300)
    assert rc == 0 and rco == 0 and r < 1e-10 and no < 300
    assert rel(U, Uo) < 1e-7
    if kw.get("precision"):
        s64 = gputo.Solver(nelx, nely, nelz, nl, preset=preset, nswp=kw.get("nswp", 0))
        n64 = s64.solve(Ke, F, CX, fixed, 1e-10, 300)[2]
        s64.close()
        print("iterations", n64, n, flush=True)
        assert n <= n64 + (40 if kw.get("l0_kernel") == 3 else 2)
    else:
        r10 = s.solve(Ke, F, CX, fixed, 1e-10, 10)[1]
        ro10 = oracle.mgcg(Ke, F, CX, fixed, nelx, nely, nelz, nl, 1e-10, 10, preset=preset, nswp=2)[1]
        print("residuals", ro10, r10, flush=True)
        assert abs(r10 - ro10) <= 1e-6 * ro10
    s.close()


@pytest.mark.parametrize("kind", ["classes", "full"])
@pytest.mark.parametrize("kw", [dict(), dict(preset=1), dict(preset=2), dict(homog_sequential=1), dict(precision=1),
                                dict(precision=2, l0_kernel=3)])
def test_periodic_cell(gputo, kw, kind):
    """The fold and image kernels around the operator."""
    import periodic_oracle

    shape = (12, 8, 16)
    print("case", kw, kind, flush=True)
    CX = 0.01 + 0.99 * np.random.default_rng(85).uniform(size=shape[0] * shape[1] * shape[2])
    Ke = element(gputo, kind, 1e-9)
    s = gputo.Solver(*shape, 3, periodic=True, **kw)
    C, r, n, _ = s.homogenize(Ke, CX, 1e-10, 500)
    s.close()
    Co, _ = periodic_oracle.homogenize(Ke, CX, *shape)
    assert (r < 1e-10).all()
    assert rel(C, Co) < 1e-8


@pytest.mark.parametrize("mesh", [(2, 2, 2), (24, 12, 12), (7, 33, 5)])
def test_matvec_without_allocation(gputo, oracle, mesh):
    """Through the node mask, twice with different fixed DOFs (the mask of the first
    call is cleared), some of them outside the mesh, which are skipped."""
    lib = gputo.load()
    print("case", mesh, flush=True)
    _, F, CX, fixed = cantilever_case(*mesh, seed=86)
    Ke = element(gputo, "classes", 1e-3)
    u = np.random.default_rng(87).uniform(-1, 1, F.size)
    dev = Dev()
    try:
        dCX, du, dy = dev.put(CX), dev.put(u), dev.put(np.full(F.size, np.nan))
        for fx in ((fixed - 1).astype(np.int32), np.array([-1, 5, F.size - 1, F.size], dtype=np.int32)):
            rc = lib.gputo_matvec_f64_noalloc(*mesh, Ke.ctypes.data_as(ctypes.c_void_p), dCX, du, dev.put(fx), len(fx),
                                              dy, None)
            assert rc == 0
            dev.sync()
            y = dev.get(dy, F.size)
            inside = fx[(fx >= 0) & (fx < F.size)]
            assert rel(y, oracle.matvec0(Ke, CX, u, inside + 1.0, *mesh)) < 1e-13
            assert not y[inside].any()
    finally:
        dev.free()
