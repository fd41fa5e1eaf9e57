"""The PCG's residual test inside the V-cycle's first level-0 sweep (a block of
its own) and as a launch: iteration counts and relative residuals against the
oracle's, where the iteration limit ends the solve before, at and after
convergence.

The residual after a few iterations agrees to the rounding of the two summation
orders times the growth of a CG iteration: 1e-6 of its value in FP64.  With an
FP32 V-cycle the iterates differ by FP32 rounding (6e-8) times the same growth:
1e-2.
"""
import numpy as np
import pytest

from conftest import cantilever_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("preset,precision,kw", [(0, 0, {}), (1, 0, {}), (2, 0, {}), (0, 1, {}), (0, 1, dict(graph_vcycles=1)),
                                                 (0, 2, dict(l0_kernel=5)), (0, 1, dict(mixed_npre0=1, mixed_npost0=3))])
def test_iteration_limits(gputo, oracle, preset, precision, kw):
    mesh = (16, 8, 8, 3)
    print("case", mesh, preset, precision, kw, flush=True)
    Ke, F, CX, fixed = cantilever_case(*mesh[:3], seed=71)
    s = gputo.Solver(*mesh, preset=preset, precision=precision, **kw)
    _, relres, nit, rc = s.solve(Ke, F, CX, fixed, 1e-8, 500)
    assert rc == 0 and relres < 1e-8 and 2 < nit < 500
    for maxit in (1, 2, nit, nit + 1):
        U, r, n, rc = s.solve(Ke, F, CX, fixed, 1e-8, maxit)
        assert rc == 0 and n == min(maxit, nit)
        assert (r < 1e-8) == (maxit > nit)  # nit counts the iterations before the converged one
        if maxit <= 2 and not kw.get("mixed_npre0"):
            oracle.lib().or_set_nswp(2)
            Uo, ro, no, rco = oracle.mgcg(Ke, F, CX, fixed, *mesh, 1e-8, maxit, preset=preset)
            if precision == 0:
                assert abs(r - ro) <= 1e-6 * ro
            elif kw.get("l0_kernel") != 5:
                assert abs(r - ro) <= 1e-2 * ro
        if maxit > nit:
            assert r == relres
    s.close()
