"""What cpfem_solve_mg does on boxes where the Jacobi solve is the faster one: no multigrid work at all,
seen in the library's launch counters, and the Jacobi solve's result to the last bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _system(n, h, held):
    """Newton system of an FCC polycrystal box of n elements of proportions h, a little past yield."""
    import cpfem_amd as C
    from cpfem_amd import configs
    from cpfem_amd.solver import bc_x0
    rng = np.random.default_rng(0)
    L = np.asarray(n, dtype=float) * np.asarray(h, dtype=float)
    L /= L.max()
    m = C.box_mesh(*n, *L)
    at = lambda d, v: (lambda p: np.isclose(p[d], v, atol=1e-9))  # noqa: E731
    zero = lambda p: np.zeros_like(p[0])  # noqa: E731
    top = lambda p: np.full_like(p[0], 9e-4 * L[2])  # noqa: E731
    if held:
        info = [[at(2, 0.0)] * 3 + [at(2, L[2])] * 3, [0, 1, 2, 0, 1, 2], [zero] * 5 + [top]]
    else:
        info = [[at(0, 0.0), at(1, 0.0), at(2, 0.0), at(2, L[2])], [0, 1, 2, 2], [zero, zero, zero, top]]
    quat = rng.normal(size=(40, 4))
    quat /= np.linalg.norm(quat, axis=1, keepdims=True)
    cells = m.cells_dict["hexahedron"]
    prob = C.CrystalPlasticity(C.Mesh(m.points, cells), dirichlet_bc_info=info, material=configs.config2(n=4).material,
                               additional_info=(quat, rng.integers(0, 40, len(cells))))
    prob.dt = 0.9
    dofs = torch.as_tensor((np.array(m.points) * np.array([-3e-4, -3e-4, 8e-4])).ravel(), device="cuda")
    res, mat = prob.assemble(dofs)
    return prob, mat.clone(), -res, bc_x0(prob, dofs)


def _launches(prob, solve):
    """solve()'s result and the launches of the multigrid classes in it."""
    from cpfem_amd import _native as N
    L, h, n = prob.ctx._lib, prob.ctx.h, len(N.PROF_CLASSES)
    N.check(L.cpfem_profile(h, 1, 1))
    x = solve()
    ms, la, ti = (ctypes.c_double * n)(), (ctypes.c_int64 * n)(), (ctypes.c_int64 * n)()
    N.check(L.cpfem_profile_read(h, n, ms, la, ti))
    N.check(L.cpfem_profile(h, 0, 1))
    return x, {c: la[k] for k, c in enumerate(N.PROF_CLASSES) if c.startswith("mg_")}


@pytest.mark.parametrize("n, h, held", [((24, 24, 6), (1, 1, 1), True), ((16, 16, 16), (1, 1, 0.2), True),
                                        ((16, 16, 16), (1, 1, 7), False)])
def test_no_multigrid_work_where_the_jacobi_solve_is_faster(n, h, held):
    from cpfem_amd.solver import krylov_solve, multigrid_solve
    prob, mat, b, x0 = _system(n, h, held)
    xj = krylov_solve(prob, mat, b, x0)
    x, launches = _launches(prob, lambda: multigrid_solve(prob, mat, b, x0))
    print(n, h, held, launches, prob.solver_info[-1]["iterations"], flush=True)
    assert not any(launches.values())
    assert torch.equal(x, xj)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n, h", [((24, 24, 6), (1, 1, 0.3)), ((80, 80, 3), (1, 1, 1)), ((24, 24, 7), (1, 1, 0.5))])
def test_thin_boxes_whose_second_level_has_a_lower_spectrum(n, h, precision):
    """The second level's lambda_max is 1.13 to 1.2 times below the finest one's, beyond what the
    polynomial's range allows for: the range has to be the finest level's.  The bars are those of the other
    comparisons with the Jacobi solve: |r| <= 1e-11 (|b| + |r0|) where both solves stop at 1e-12."""
    import cpfem_amd as C
    from cpfem_amd.solver import krylov_solve, multigrid_solve
    prob, mat, b, x0 = _system(n, h, False)
    opts = {"krylov_tol": 1e-12, "krylov_atol": 1e-14, "precision": precision}
    xj = krylov_solve(prob, mat, b, x0, opts).cpu().numpy()
    x = multigrid_solve(prob, mat, b, x0, opts).cpu().numpy()
    k = prob.solver_info[-1]["iterations"]
    A = C.BlockEllMatrix(prob.ctx, mat).to_scipy()
    bh = b.cpu().numpy()
    r, bar = np.linalg.norm(A @ x - bh), 1e-11 * (np.linalg.norm(bh) + np.linalg.norm(bh - A @ x0.cpu().numpy()))
    print(n, h, precision, k, f"|Ax - b| {r:.2e} (bar {bar:.2e})", flush=True)
    assert 0 < k <= 30
    assert r <= bar
    assert np.linalg.norm(x - xj) <= 1e-7 * np.linalg.norm(xj)


@pytest.mark.parametrize("n, h", [((32, 32, 4), (1, 1, 0.5)), ((2, 2, 60), (1, 1, 1.4))])
def test_thin_boxes_whose_second_level_is_no_coarse_form(n, h):
    """Where the second level's lambda_max lies further below, no iteration is begun."""
    from cpfem_amd.solver import krylov_solve, multigrid_solve
    prob, mat, b, x0 = _system(n, h, False)
    xj = krylov_solve(prob, mat, b, x0)
    x, launches = _launches(prob, lambda: multigrid_solve(prob, mat, b, x0))
    assert launches["mg_setup"] > 0 and launches["mg_fine"] == 0
    assert torch.equal(x, xj)


def test_an_attempt_in_vain_leaves_nothing_behind():
    """A system that the estimates let through and multigrid does not solve: the Jacobi solve starts from x0."""
    from cpfem_amd.solver import krylov_solve, multigrid_solve
    prob, mat, b, x0 = _system((3, 20, 20), (1, 1, 4), True)
    xj = krylov_solve(prob, mat, b, x0)
    x, launches = _launches(prob, lambda: multigrid_solve(prob, mat, b, x0))
    assert launches["mg_fine"] > 0
    assert prob.solver_info[-1]["iterations"] == prob.solver_info[-2]["iterations"] > 60
    assert torch.equal(x, xj)


def test_new_dirichlet_dofs_are_looked_at_again():
    """A box with symmetry planes, then held on two faces, then as before."""
    from cpfem_amd.solver import multigrid_solve
    prob, mat, b, x0 = _system((24, 24, 6), (1, 1, 1), False)
    symmetry = prob.fes[0].dirichlet_bc_info
    held_prob, hmat, hb, hx0 = _system((24, 24, 6), (1, 1, 1), True)
    held = held_prob.fes[0].dirichlet_bc_info
    x, launches = _launches(prob, lambda: multigrid_solve(prob, mat, b, x0))
    assert launches["mg_fine"] > 0
    prob.fes[0].update_Dirichlet_boundary_conditions(held)
    xh, launches = _launches(prob, lambda: multigrid_solve(prob, hmat, hb, hx0))
    assert not any(launches.values())
    assert torch.equal(xh, multigrid_solve(held_prob, hmat, hb, hx0))
    prob.fes[0].update_Dirichlet_boundary_conditions(symmetry)
    y, launches = _launches(prob, lambda: multigrid_solve(prob, mat, b, x0))
    assert launches["mg_fine"] > 0
    assert torch.equal(x, y)
