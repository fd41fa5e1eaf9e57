"""Host arrays that go to the device in one chunk (small), in chunks of one
thread and of several threads, with a ragged last chunk: bytes unchanged, and a
NaN or an infinity anywhere in an array is found."""
import numpy as np
import pytest

from conftest import cantilever_case

pytestmark = pytest.mark.gpu

MESHES = [(8, 4, 4, 3), (56, 40, 40, 4), (96, 88, 72, 4)]  # 0.1, 3.4 and 24 MB


@pytest.mark.parametrize("mesh", MESHES)
def test_design_arrays_unchanged(gputo, mesh):
    nelx, nely, nelz, nl = mesh
    print("case", mesh, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=1)
    rng = np.random.default_rng(2)
    s = gputo.Solver(nelx, nely, nelz, nl)
    try:
        for nfd in (fixed.size, fixed.size - 3, fixed.size):  # the loop's buffers are reused
            x0 = rng.uniform(0.1, 1.0, s.nel)
            loop = gputo.TopOpt(s, Ke, x0, F, fixed[:nfd])
            x, xp, U = loop.state()
            loop.close()
            assert np.array_equal(x, x0) and np.array_equal(xp, x0) and not U.any()
    finally:
        s.close()


@pytest.mark.parametrize("mesh", MESHES)
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_nonfinite_is_found(gputo, mesh, value):
    nelx, nely, nelz, nl = mesh
    print("case", mesh, value, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=1)
    s = gputo.Solver(nelx, nely, nelz, nl)
    try:
        for a, at in ((0, 0), (0, -1), (0, CX.size // 2), (1, 0), (1, -1), (1, F.size // 2)):
            arrays = [CX.copy(), F.copy()]
            arrays[a][at] = value
            U, relres, nit, rc = s.solve(Ke, arrays[1], arrays[0], fixed, 1e-6, 1)
            assert rc == -3 and not U.any()
        F2 = F.copy()
        F2[-1] = 1e100  # finite, and its square too
        assert s.solve(Ke, F2, CX, fixed, 1e-6, 1)[3] != -3
    finally:
        s.close()
