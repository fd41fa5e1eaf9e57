"""The mgcg9 engine (GPUTO_PRESET_MGCG9, Homogenization/QNC/mgcg9.cu)
against the oracle's restatement: coarse element scales bit-exact (same
summation order), fixed lists bit-exact, diagonals 1e-14, and the solve
(nit within one, U to 1e-8, compliance to 1e-9) for several nswp, with the
factored coarsest level and with the smoothed one (coarsest >= 20000 DOFs).
"""
import numpy as np
import pytest

from conftest import cantilever_case

pytestmark = pytest.mark.gpu
MGCG9 = 2


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("mesh", [(16, 8, 8, 3), (32, 16, 16, 4)])
def test_mgcg9_hierarchy(gputo, oracle, mesh):
    nelx, nely, nelz, nl = mesh
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=51, kind="perturbed")
    s = gputo.Solver(nelx, nely, nelz, nl, preset=MGCG9)
    s.setup(Ke, CX, fixed)
    for l in range(nl):
        assert np.array_equal(s.level_cx(l), oracle.level_cx(Ke, CX, fixed, nelx, nely, nelz, nl, l))
        _, ad, fd = s.level_matrices(l)
        _, ado, fdo = oracle.level_data(Ke, CX, fixed, nelx, nely, nelz, nl, l, preset=MGCG9)
        assert np.array_equal(fd, fdo)
        assert rel(ad, ado) < 1e-14
    s.close()


@pytest.mark.parametrize("nswp", [1, 2, 4])
@pytest.mark.parametrize("mesh,kind", [((16, 8, 8, 3), "smooth"), ((32, 16, 16, 4), "perturbed"),
                                       ((48, 24, 24, 4), "smooth")])
def test_mgcg9_solve_matches_oracle(gputo, oracle, mesh, kind, nswp):
    nelx, nely, nelz, nl = mesh
    print("case", mesh, kind, nswp, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=52, kind=kind)
    s = gputo.Solver(nelx, nely, nelz, nl, preset=MGCG9, nswp=nswp)
    if nswp == 1 and kind == "perturbed":
        # one sweep each way with omega 0.33 leaves this preconditioner
        # indefinite: the oracle stalls (relres 2.3e-4 after 400 iterations),
        # so the two are compared over the same 20 capped iterations
        Uo, ro, no, rco = oracle.mgcg(Ke, F, CX, fixed, nelx, nely, nelz, nl, 1e-12, 20, preset=MGCG9, nswp=nswp)
        U, r, n, rc = s.solve(Ke, F, CX, fixed, 1e-12, 20)
        assert rc == 0 and rco == 0 and n == no == 20
        assert abs(r - ro) <= 1e-7 * ro
        assert rel(U, Uo) < 1e-7
    else:
        Uo, ro, no, rco = oracle.mgcg(Ke, F, CX, fixed, nelx, nely, nelz, nl, 1e-9, 400, preset=MGCG9, nswp=nswp)
        U, r, n, rc = s.solve(Ke, F, CX, fixed, 1e-9, 400)
        assert rc == 0 and rco == 0
        assert no < 400, "the oracle converges on every other case (16-86 iterations)"
        assert abs(n - no) <= 1 and r < 1e-9
        assert rel(U, Uo) < 1e-7
        assert abs(F @ U - F @ Uo) <= 1e-8 * abs(F @ Uo)
    s.close()


def test_mgcg9_smoothed_coarsest_level(gputo, oracle):
    """nl = 2 at 64x32x32: the coarsest level has 3*33*17*17 = 28611 >= 20000
    DOFs, so it gets 10*nswp Jacobi sweeps from its previous iterate instead
    of a Cholesky solve.  That preconditioner changes between iterations and
    the reference's CG does not converge with it here, so the two are
    compared over the same 6 iterations (the level starts from zero)."""
    nelx, nely, nelz, nl = 64, 32, 32, 2
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=53, kind="smooth")
    Uo, ro, no, rco = oracle.mgcg(Ke, F, CX, fixed, nelx, nely, nelz, nl, 1e-12, 6, preset=MGCG9, nswp=2)
    s = gputo.Solver(nelx, nely, nelz, nl, preset=MGCG9, nswp=2)
    U, r, n, rc = s.solve(Ke, F, CX, fixed, 1e-12, 6)
    assert rc == 0 and rco == 0 and n == no == 6
    assert abs(r - ro) <= 1e-8 * ro
    assert rel(U, Uo) < 1e-9
    s.close()


def test_mgcg9_matlab_interface(gputo, oracle):
    nelx, nely, nelz, nl = 16, 8, 8, 3
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=54, kind="smooth")
    U = np.zeros_like(F)
    cgres, cgiters = gputo.mgcg9(Ke, F, U, CX, fixed, len(fixed), nelx, nely, nelz, nl, 1e-9, 300, 3, 0, 0.3,
                                 1.0, 1.0, 1.0)
    Uo, ro, no, _ = oracle.mgcg(Ke, F, CX, fixed, nelx, nely, nelz, nl, 1e-9, 300, preset=MGCG9, nswp=3)
    assert abs(cgiters - no) <= 1 and cgres < 1e-9
    assert rel(U, Uo) < 1e-7
    gputo.release_handles()


def test_coarse_solve_without_a_factor_is_refused(gputo):
    """A smoothed coarsest level has no factor to solve with."""
    nelx, nely, nelz, nl = 64, 32, 32, 2
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=55, kind="smooth")
    s = gputo.Solver(nelx, nely, nelz, nl, preset=MGCG9)
    s.setup(Ke, CX, fixed)
    with pytest.raises(gputo.GputoError):
        s.coarse_solve(np.zeros(3 * 33 * 17 * 17))
    s.close()
