"""The coarsest solve, whose factorisation is split at the middle plane from five
planes and four 32-row tiles on, against numpy's dense solve of the assembled
matrix.

Coarsest grids (nodes): 7x7x3 (parts of 189 DOFs in 192 rows), 8x5x5 (parts of
four and three planes), 5x5x5 (two planes to a part), 17x4x5 (many steps),
9x9x9 (band 275), 5x3x3 (five tiles), 5x2x2 and 3x3x3 (too few rows to split),
4x9x9 (too few planes, wide band) and, with the decoupled fixed DOFs of the
mgcg9 engine, 12x8x10 and 8x5x5.  Tolerance as for the other coarsest solves:
the conditioning of the penalised matrix (1e-9)."""
import numpy as np
import pytest

from conftest import cantilever_case

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("coarse", [(6, 6, 2), (7, 4, 4), (4, 4, 4), (16, 3, 4), (8, 8, 8), (4, 2, 2), (4, 1, 1),
                                    (2, 2, 2), (3, 8, 8)])
def test_split_coarse_solve(gputo, oracle, coarse):
    cx, cy, cz = coarse
    nelx, nely, nelz = 2 * cx, 2 * cy, 2 * cz
    print("case", coarse, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=8)
    s = gputo.Solver(nelx, nely, nelz, 2)
    try:
        s.setup(Ke, CX, fixed)
        A, _, fd = s.level_matrices(1)
        AQ = oracle.assemble(A, cx, cy, cz)
        rng = np.random.default_rng(9)
        for _ in range(2):
            b = rng.uniform(-1, 1, AQ.shape[0])
            b[(fd - 1).astype(int)] = 0.0
            x = s.coarse_solve(b)
            xr = np.linalg.solve(AQ, b)
            xr[(fd - 1).astype(int)] = 0.0
            assert rel(x, xr) < 1e-9
    finally:
        s.close()


@pytest.mark.parametrize("mesh,nl", [((44, 28, 36), 3), ((28, 16, 16), 3)])
def test_split_decoupled_fixed_dofs(gputo, oracle, mesh, nl):
    """One V-cycle of the mgcg9 engine, whose fixed rows and columns are
    decoupled while the matrix is assembled."""
    nelx, nely, nelz = mesh
    print("case", mesh, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=10)
    r = np.random.default_rng(11).uniform(-1, 1, F.size)
    r[(fixed - 1).astype(int)] = 0.0
    s = gputo.Solver(nelx, nely, nelz, nl, preset=2)
    try:
        z = s.vcycle(Ke, CX, fixed, r)
    finally:
        s.close()
    oracle.lib().or_set_nswp(2)
    zo = oracle.vcycle_once(Ke, CX, fixed, nelx, nely, nelz, nl, r, preset=2)
    assert rel(z, zo) < 1e-9


@pytest.mark.parametrize("mesh", [(2, 2, 2, 2), (4, 4, 4, 2), (8, 4, 4, 2), (12, 8, 8, 2), (14, 12, 10, 2), (16, 10, 12, 2)])
def test_whole_inverse(gputo, oracle, mesh):
    """Coarsest solves by the whole inverse: one tile, three without the split, two
    parts of different lengths, 1024 entries (the most), and the two products just
    above; FP32 vectors through a mixed solve.  Tolerance of the other coarsest
    solves."""
    nelx, nely, nelz, nl = mesh
    print("case", mesh, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=8)
    s = gputo.Solver(nelx, nely, nelz, nl)
    s.setup(Ke, CX, fixed)
    A, _, fd = s.level_matrices(nl - 1)
    AQ = oracle.assemble(A, nelx // 2, nely // 2, nelz // 2)
    b = np.random.default_rng(9).uniform(-1, 1, AQ.shape[0])
    b[(fd - 1).astype(int)] = 0.0
    x = s.coarse_solve(b)
    xr = np.linalg.solve(AQ, b)
    xr[(fd - 1).astype(int)] = 0.0
    assert np.abs(x - xr).max() < 1e-9 * np.abs(xr).max()
    U, _, _, rc = s.solve(Ke, F, CX, fixed, 1e-10, 500)
    s.close()
    m = gputo.Solver(nelx, nely, nelz, nl, precision=1)
    Um, _, _, rcm = m.solve(Ke, F, CX, fixed, 1e-10, 500)
    m.close()
    assert rc == 0 and rcm == 0 and np.abs(Um - U).max() < 1e-8 * np.abs(U).max()


@pytest.mark.parametrize("coarse", [(9, 2, 2), (7, 2, 2), (5, 2, 2), (6, 2, 2), (1, 1, 1)])
def test_block_columns_in_pairs(gputo, oracle, coarse):
    """Parts of 5 and 4, 4 and 3, 3 and 2, 3 and 3 block columns (pairs, and a last
    one alone, in one part or both), and a matrix of one."""
    nelx, nely, nelz = (2 * c for c in coarse)
    print("case", coarse, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=8)
    s = gputo.Solver(nelx, nely, nelz, 2)
    s.setup(Ke, CX, fixed)
    A, _, fd = s.level_matrices(1)
    AQ = oracle.assemble(A, *coarse)
    b = np.random.default_rng(9).uniform(-1, 1, AQ.shape[0])
    b[(fd - 1).astype(int)] = 0.0
    x = s.coarse_solve(b)
    s.close()
    xr = np.linalg.solve(AQ, b)
    xr[(fd - 1).astype(int)] = 0.0
    assert rel(x, xr) < 1e-9
