"""The design loop's filter and optimality-criteria bisection where they can go
wrong: every compiled half width and the general one, meshes narrower than the
window, brackets that need more than one batch of bisection passes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", [(8, 4, 4, 2), (4, 2, 6, 2), (24, 10, 14, 2)])
@pytest.mark.parametrize("rmin", [1.0, 1.5, 2.0, 2.9, 3.2, 4.0, 4.5, 6.1])
def test_filter_widths(gputo, oracle, mesh, rmin):
    """Same products in the same order as the oracle's filter: 1e-14."""
    nelx, nely, nelz, nl = mesh
    x = np.random.default_rng(16).uniform(0, 1, nelx * nely * nelz)
    s = gputo.Solver(nelx, nely, nelz, nl)
    try:
        y, yo = s.filter(x, rmin), oracle.imfilter(x, nelx, nely, nelz, rmin)
    finally:
        s.close()
    assert np.abs(y - yo).max() < 1e-14 * np.abs(yo).max()


@pytest.mark.parametrize("volfrac,x0", [(0.12, 0.12), (0.8, 0.3), (0.05, 0.6)])
def test_bisection_brackets(gputo, oracle, volfrac, x0):
    """An ordinary bracket, a volume out of reach from below (the multiplier runs
    to zero, some 1075 halvings) and from above (to the upper end)."""
    nelx, nely, nelz, nl = 12, 6, 6, 2
    print("case", volfrac, x0, flush=True)
    Ke, F, fixed = gputo.cantilever(nelx, nely, nelz)
    x = np.full(nelx * nely * nelz, x0)
    rmin = np.sqrt(3.0)
    s = gputo.Solver(nelx, nely, nelz, nl)
    run = gputo.TopOpt(s, Ke, x, F, fixed, volfrac=volfrac, penal=3.0, rmin=rmin, eta=0.4, beta=2.0, move=0.2, ft=1,
                       cg_tol=1e-12, cg_maxit=400)
    st = oracle.DesignState(nelx, nely, nelz, x, eta=0.4)
    try:
        g = run.iterate()
        o = oracle.design_iter(st, Ke, F, fixed, nl, 1e-12, 400, volfrac, 3.0, rmin, 1, 2.0, 0.2)
        assert g["status"] == 0 and o["rc"] == 0
        # the multiplier's bracket is 1e-4 wide, the same halvings on both sides
        xg = run.state()[0]
        assert np.abs(xg - st.x).max() < 1e-8
    finally:
        run.close()
        s.close()
