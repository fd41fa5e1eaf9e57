"""The coarsest factor where a step has more tiles than fit the chip together: the
panel once per row tile, then the trailing band (k_chol_update), down to the
steps that are small again.  Against numpy's dense solve of the assembled matrix.

Coarsest grids (nodes): 5x15x15 (split at the middle plane: two parts at once,
band 725, an odd number of trailing tiles), 4x19x19 (one part, band 1145) and
6x16x15; a periodic 7^3 cell, whose matrix has no band.  Tolerance as for the
other coarsest solves: the conditioning of the penalised matrix (1e-9)."""
import numpy as np
import pytest

from conftest import cantilever_case

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("coarse", [(4, 14, 14), (3, 18, 18), (5, 15, 14)])
def test_wide_band(gputo, oracle, coarse):
    cx, cy, cz = coarse
    print("case", coarse, flush=True)
    Ke, F, CX, fixed = cantilever_case(2 * cx, 2 * cy, 2 * cz, seed=8)
    s = gputo.Solver(2 * cx, 2 * cy, 2 * cz, 2)
    s.setup(Ke, CX, fixed)
    A, _, fd = s.level_matrices(1)
    AQ = oracle.assemble(A, cx, cy, cz)
    fx = (fd - 1).astype(int)
    b = np.random.default_rng(9).uniform(-1, 1, AQ.shape[0])
    b[fx] = 0.0
    x = s.coarse_solve(b)
    s.close()
    xr = np.linalg.solve(AQ, b)
    xr[fx] = 0.0
    assert rel(x, xr) < 1e-9


def test_dense_periodic_cell(gputo):
    c = 7
    n = 2 * c
    Ke = gputo.ke0_h8()
    CX = np.random.default_rng(10).uniform(0.1, 1.0, n ** 3)
    corners = [(i * (n + 1) + k) * (n + 1) + j for i in (0, n) for k in (0, n) for j in (0, n)]
    fixed = np.array([3.0 * q + d + 1 for q in corners for d in range(3)])
    s = gputo.Solver(n, n, n, 2, periodic=True)
    s.setup(Ke, CX, fixed)
    A, _, fd = s.level_matrices(1)
    # the masters' matrix: element nodes wrapped, the pinned node decoupled
    node = lambda i, k, j: (i % c * c + k % c) * c + j % c  # noqa: E731
    ie, je, ke = (0, 1, 1, 0, 0, 1, 1, 0), (0, 0, 1, 1, 0, 0, 1, 1), (0, 0, 0, 0, 1, 1, 1, 1)
    K = np.zeros((3 * c ** 3, 3 * c ** 3))
    for i in range(c):
        for k in range(c):
            for j in range(c):
                d = np.concatenate([3 * node(i + ie[a], k + ke[a], j + je[a]) + np.arange(3) for a in range(8)])
                K[np.ix_(d, d)] += A[(i * c + k) * c + j]
    K[:3] = 0.0
    K[:, :3] = 0.0
    K[range(3), range(3)] = 1e10
    f = np.random.default_rng(11).uniform(-1, 1, (c, c, c, 3))
    f[0, 0, 0] = 0.0
    b = np.zeros((c + 1, c + 1, c + 1, 3))
    b[:c, :c, :c] = f
    x = s.coarse_solve(b.ravel()).reshape(b.shape)[:c, :c, :c]
    s.close()
    assert rel(x.ravel(), np.linalg.solve(K, f.ravel())) < 1e-9
