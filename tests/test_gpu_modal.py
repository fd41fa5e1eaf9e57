"""The matrix-free operators in the modal basis (csrc/modal.hip) at the edges
of their tiling, against the oracle's element products (multAV0c / defect0c /
Jacobc, Cantilever/TOP3D125MGCGCUDA/mgcg1.cu:941-997,1190-1264): one element
per direction and level, rows longer and shorter than a wave, several strips
along j, chunks of a plane and layer groups along i, remainders in each.

Tolerances relative to max|y|: FP64 1e-13 (summation order only), FP32 2e-6
(FP32 rounding of the operands and sums), as the other operator tests.
"""
import numpy as np
import pytest

from conftest import cantilever_case

pytestmark = pytest.mark.gpu

OMEGA, PRERELAX = 0.48, 0.7  # Jacobc, preRelc of the reference smoother

MESHES = [(2, 2, 2, 2), (2, 62, 2, 2), (4, 128, 2, 2), (2, 2, 130, 2), (130, 2, 4, 2), (12, 36, 20, 3), (20, 68, 44, 3),
          (72, 56, 40, 4), (112, 96, 48, 5)]


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def references(Ku, u, f, ad, fx):
    """mode -> reference of gputo_level_apply from the product Ku(u)."""
    out = {}
    for mode in range(5):
        uu = PRERELAX * f / ad if mode in (3, 4) else u
        y = Ku(uu)
        r = f - y
        r[fx] = 0.0
        if mode == 0:
            y[fx] = 0.0
            out[mode] = y
        elif mode in (1, 4):
            out[mode] = r
        else:
            out[mode] = (1 - OMEGA) * uu + OMEGA * (r + ad * uu) / ad
    return out


def check_levels(gputo, oracle, mesh, levels):
    nelx, nely, nelz, nl = mesh
    print("case", mesh, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=61, kind="smooth")
    s = gputo.Solver(nelx, nely, nelz, nl, precision=1)
    s.setup(Ke, CX, fixed)
    rng = np.random.default_rng(62)
    for level in levels:
        if level == 0:
            ad, fx = oracle.prepad0(Ke, CX, nelx, nely, nelz), (fixed - 1).astype(np.int64)

            def Ku(v):
                return oracle.matvec0(Ke, CX, v, np.zeros(0), nelx, nely, nelz)
        else:
            A, ad, fd = oracle.level_data(Ke, CX, fixed, nelx, nely, nelz, nl, 1)
            fx = fd.astype(np.int64) - 1

            def Ku(v):
                return oracle.matvec_el(A, v, np.zeros(0), nelx // 2, nely // 2, nelz // 2)
        u, f = rng.uniform(-1, 1, ad.size), rng.uniform(-1, 1, ad.size)
        ref = references(Ku, u, f, ad, fx)
        for mode in range(5):
            for fp32, tol in ((False, 1e-13), (True, 2e-6)):
                y = s.level_apply(level, 1 + level, mode, u, f, fp32=fp32)
                assert rel(y, ref[mode]) < tol, (level, mode, fp32, rel(y, ref[mode]))
                assert np.array_equal(y, s.level_apply(level, 1 + level, mode, u, f, fp32=fp32))
    s.close()


@pytest.mark.parametrize("mesh", MESHES)
def test_modal_operators_vs_oracle(gputo, oracle, mesh):
    check_levels(gputo, oracle, mesh, range(1 if mesh[3] < 3 else 2))


@pytest.mark.parametrize("mesh", [(16, 8, 8, 3), (48, 48, 48, 4), (88, 40, 56, 4), (120, 56, 56, 4)])
def test_level1_with_a_wave_group_per_layer(gputo, oracle, mesh):
    """Level-1 grids whose blocks own one, two, three (a last block of fewer) and,
    FP32 only, six node layers with a wave per element layer."""
    check_levels(gputo, oracle, mesh, [1])


@pytest.mark.parametrize("mesh", [(4, 6, 8, 2), (20, 68, 44, 3)])
def test_modal_keeps_non_finite_values_local(gputo, mesh):
    """A NaN or infinity at a node reaches the 27 nodes around it and no other
    (elements outside the mesh are worked on, but read nothing)."""
    nelx, nely, nelz, nl = mesh
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=63)
    s = gputo.Solver(nelx, nely, nelz, nl)
    for i, k, j in ((nelx, nelz, nely), (1, 1, 0), (nelx // 2, nelz, 0), (0, 0, nely)):
        u = np.zeros((nelx + 1, nelz + 1, nely + 1, 3))
        u[i, k, j, 1] = np.nan if j else np.inf
        y = s.matvec(Ke, CX, u.ravel(), fixed).reshape(u.shape)
        bad = ~np.isfinite(y).all(axis=-1)
        near = np.zeros_like(bad)
        near[max(i - 1, 0):i + 2, max(k - 1, 0):k + 2, max(j - 1, 0):j + 2] = True
        near[0] = False  # the fixed face
        assert np.array_equal(bad, near)
        assert not y[~near].any()
    s.close()


@pytest.mark.parametrize("kernel,tol", [(1, 2e-6), (2, 2e-6), (3, 1e-4), (4, 2e-6)])
def test_other_element_matrices_take_the_general_kernels(gputo, oracle, kernel, tol):
    """A Ke0 without the isotropic modal form: the node-gather and the MFMA kernels."""
    nelx, nely, nelz, nl = 40, 20, 12, 3
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=64, kind="smooth")
    E = np.random.default_rng(65).uniform(-1, 1, (24, 24)) * 1e-3
    Ke = Ke + (E + E.T)
    s = gputo.Solver(nelx, nely, nelz, nl, precision=2, l0_kernel=kernel)
    u = np.random.default_rng(66).uniform(-1, 1, s.ndof)
    yo = oracle.matvec0(Ke, CX, u, fixed, nelx, nely, nelz)
    assert rel(s.matvec_mixed(kernel, Ke, CX, u, fixed), yo) < tol
    assert rel(s.matvec(Ke, CX, u, fixed), yo) < 1e-13
    s.close()


@pytest.mark.parametrize("cell", [(4, 4, 4), (8, 136, 4), (4, 24, 68), (68, 4, 20)])
def test_periodic_form_is_translation_invariant(gputo, cell):
    """The periodic form of the kernels over cells that need one and several
    strips, chunks and layer groups: a cell moved by half its size in each
    direction has the same tensor (1e-8, the CG tolerance), and images hold
    their masters' values bit for bit."""
    nx, ny, nz = cell
    rng = np.random.default_rng(67)
    x = 0.2 + 0.8 * rng.uniform(size=(nx, nz, ny))
    Ke = gputo.ke0_h8()
    s = gputo.Solver(nx, ny, nz, 2, periodic=True)
    C, _, _, chi = s.homogenize(Ke, x.ravel(), 1e-10, 400, fields=True)
    C2 = s.homogenize(Ke, np.roll(x, (nx // 2, nz // 2, ny // 2), (0, 1, 2)).ravel(), 1e-10, 400)[0]
    assert np.abs(C - C2).max() < 1e-8 * np.abs(C).max()
    u = chi.reshape(6, nx + 1, nz + 1, ny + 1, 3)
    assert np.array_equal(u[:, 0], u[:, -1])
    assert np.array_equal(u[:, :, 0], u[:, :, -1])
    assert np.array_equal(u[:, :, :, 0], u[:, :, :, -1])
    s.close()


@pytest.mark.parametrize("preset", [0, 1])
@pytest.mark.parametrize("mesh", [(16, 8, 8, 3), (4, 124, 4, 3), (4, 4, 260, 3), (260, 4, 8, 3), (12, 36, 20, 3),
                                  (16, 16, 16, 4), (72, 56, 40, 4), (112, 96, 48, 5)])
def test_correction_added_by_the_first_post_sweep(gputo, oracle, mesh, preset):
    """A V-cycle whose first sweep after a coarse correction adds it (the level-1
    operator with a wave group per layer, preset 0, and the node stencils), on
    grids at the edges of the kernels' tiles, with fixed DOFs inside the mesh and
    at its last node: the oracle's interpolation and sweeps, 1e-9 as the other
    V-cycle tests."""
    nelx, nely, nelz, nl = mesh
    print("case", mesh, preset, flush=True)
    Ke, F, CX, face = cantilever_case(nelx, nely, nelz, seed=65)
    last = F.size
    fixed = np.unique(np.concatenate([face, [last - 1, last, 3 * (last // 3 // 2) + 2]])).astype(np.float64)
    s = gputo.Solver(nelx, nely, nelz, nl, preset=preset)
    r = np.random.default_rng(66).uniform(-1, 1, s.ndof)
    r[(fixed - 1).astype(int)] = 0.0
    z = s.vcycle(Ke, CX, fixed, r)
    assert rel(z, oracle.vcycle_once(Ke, CX, fixed, nelx, nely, nelz, nl, r, preset=preset)) < 1e-9
    s.close()


@pytest.mark.parametrize("mesh", [(16, 8, 8, 3), (12, 36, 20, 3), (16, 16, 16, 4), (72, 56, 40, 4)])
def test_correction_added_by_the_first_post_sweep_fp32(gputo, mesh):
    """The same in FP32: the mixed solve ends at the FP64 solve's solution within
    a tenth more iterations (one at least) -- a correction that misses nodes
    costs several times as many."""
    nelx, nely, nelz, nl = mesh
    print("case", mesh, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=65)
    out = []
    for precision in (0, 1):
        s = gputo.Solver(nelx, nely, nelz, nl, precision=precision)
        U, _, nit, rc = s.solve(Ke, F, CX, fixed, 1e-10, 500)
        s.close()
        assert rc == 0
        out.append((U, nit))
    assert out[1][1] <= out[0][1] + max(1, out[0][1] // 10)
    assert rel(out[1][0], out[0][0]) < 1e-8


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("presets", [(1, 0), (2, 0), (0, 2), (0, 1)])
def test_level1_tiling_follows_the_preset(gputo, presets, precision):
    """A handle whose preset changes runs the level-1 operator of the new preset,
    with that element's own tiling: on this mesh the other element's has blocks
    of eight waves, twice what the FP64 level-1 element has room for.  A handle
    created with the new preset gives the same solution (1e-10, the solves'
    tolerance: its Galerkin level 1 has a stencil, the other one's element
    matrices) in as many iterations."""
    nelx, nely, nelz, nl = 208, 104, 32, 4
    print("case", presets, precision, flush=True)
    Ke, F, CX, fixed = cantilever_case(nelx, nely, nelz, seed=68, kind="uniform")
    s = gputo.Solver(nelx, nely, nelz, nl, preset=presets[0], precision=precision)
    s.set_params(preset=presets[1])
    U, _, n, rc = s.solve(Ke, F, CX, fixed, 1e-10, 200)
    s.close()
    assert rc == 0
    s = gputo.Solver(nelx, nely, nelz, nl, preset=presets[1], precision=precision)
    Uf, _, nf, rc = s.solve(Ke, F, CX, fixed, 1e-10, 200)
    s.close()
    assert rc == 0 and n == nf < 200
    assert rel(U, Uf) < 1e-10 if presets == (0, 1) else np.array_equal(U, Uf)


def test_long_rows_take_more_than_eight_strips(gputo, oracle):
    """Rows of 2305 nodes: ten strips in FP64 and fourteen in FP32; level 1 below them."""
    check_levels(gputo, oracle, (8, 2304, 8, 4), [0, 1])
