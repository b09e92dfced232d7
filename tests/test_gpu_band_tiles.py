"""Tiled band factorisation behind cpfem_solve_direct against scipy's sparse LU, at the shapes
where its schedule changes: a single tile, one front, two fronts with even and odd tile counts
and short last superblocks, full and nearly empty last tiles, a band of one tile, a wide band;
and a matrix whose elimination breaks down from the far end only, which one front must solve.

The bounds are those of the other sparse-LU comparison of this solver: 1e-9 without refinement,
1e-11 after two steps of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _system(nx, ny, nz):
    import cpfem_amd as C
    m = C.box_mesh(nx, ny, nz, float(nx), float(ny), float(nz))
    mesh = C.Mesh(m.points, m.cells_dict["hexahedron"])
    zero = lambda p: 0.0  # noqa: E731
    info = [[lambda p: np.isclose(p[0], 0.0, atol=1e-5), lambda p: np.isclose(p[1], 0.0, atol=1e-5),
             lambda p: np.isclose(p[2], 0.0, atol=1e-5), lambda p: np.isclose(p[2], float(nz), atol=1e-5)],
            [0, 1, 2, 2], [zero, zero, zero, lambda p: 1e-3 * nz]]
    quat = np.array([[0.9, 0.1, -0.3, 0.2]])
    prob = C.CrystalPlasticity(mesh, dirichlet_bc_info=info, additional_info=(quat / np.linalg.norm(quat), np.zeros(len(mesh.cells))),
                               material=C.CALIB_COPPER)
    prob.dt = 0.1
    prob.set_params(prob.internal_vars)
    dofs = torch.zeros(prob.fes[0].num_total_nodes * 3, dtype=torch.float64, device="cuda")
    res, mat = prob.assemble(dofs)
    b = torch.as_tensor(np.random.default_rng(nx + 10 * ny + 100 * nz).normal(size=len(res)), device="cuda")
    return prob, mat, b


def _check(prob, mat, b):
    import scipy.sparse.linalg as sla
    from cpfem_amd import BlockEllMatrix
    from cpfem_amd.solver import direct_solve
    A = BlockEllMatrix(prob.ctx, mat).to_scipy().tocsc()
    bh = b.cpu().numpy()
    lu = sla.splu(A)
    xr = lu.solve(bh)
    xr += lu.solve(bh - A @ xr)
    for refine, tol in ((0, 1e-9), (2, 1e-11), (2, 1e-11)):
        x = direct_solve(prob, mat, b, {"umfpack_solver": {"refine": refine}}).cpu().numpy()
        err = np.linalg.norm(x - xr) / np.linalg.norm(xr)
        print(f"{len(b)} rows, refine={refine}: {err:.2e}", flush=True)
        assert err < tol, (refine, err)


# rows: 24 and 60 (one tile), 192 (three full tiles), 324, 1029, thin bars of 492 and 972 rows,
# 2106 (wb = 3, odd tiles), a slab whose band is the whole matrix, 3600
@pytest.mark.parametrize("nx,ny,nz", [(1, 1, 1), (1, 1, 4), (3, 3, 3), (2, 2, 11), (6, 6, 6), (1, 1, 40), (1, 2, 53),
                                      (5, 3, 28), (12, 9, 1), (7, 5, 24), (11, 9, 9)])
def test_band_tiles_match_sparse_lu(nx, ny, nz):
    _check(*_system(nx, ny, nz))


def test_breakdown_from_the_far_end_is_solved_from_the_near_end():
    """The first diagonal entry of the last tile set to zero: its pivot vanishes when elimination
    starts there, and not after the rows before it are eliminated."""
    prob, mat, b = _system(1, 1, 44)  # 540 rows, nine tiles; row 512 is no Dirichlet row
    n = len(b)
    row = (n - 1) // 64 * 64
    node, comp = divmod(row, 3)
    slot = int(np.nonzero(prob.ctx.pattern()[1][:, node] == node)[0][0])
    entry = mat.view(-1, n)[3 * slot + comp]
    assert float(entry[row]) != 0.0
    entry[row] = 0.0
    _check(prob, mat, b)
