"""The point kernels' device branches against the oracle: one set of 512 points, repeated to batches of
every lane count that the launches choose (FCC: 4, 2, 1 lanes a point up to 48,000, up to 85,000 and
above; BCC24: 8, 4, 2, 1 up to 20,000, 48,000, 85,000 and above).  Neighbouring points, in one wave, take
different forms of the local Newton: a quarter has a rotation, one a rotation rounded to 32 bits, one a
sheared R and one m = 1; the last three are not for the crystal-frame form.

Bars: those of the oracle comparisons on smaller batches (stress 1e-10, Fp_inv and g 1e-12, slip 1e-9;
assembled vectors 1e-10 in norm).  Cotangents, whose terms carry the rate exponent 1/m = 50 once more
than the stresses: 50 x 1e-10 x 10 for the sum over slip systems."""
import numpy as np
import pytest

from helpers import FCC_304, random_states, slip_table

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

B = 512
G = np.array([[-2.6e-4, 1e-4, 0.0], [0.0, -2.4e-4, 1e-4], [1e-4, 0.0, 7e-4]])
TABLE = {12: "slip_fcc12.txt", 24: "slip_bcc24.txt"}
# point counts on each side of the lines between lane counts (whole cubes: 8 n^3)
CUBES = {12: (8, 18, 19, 21, 22), 24: (8, 13, 14, 18, 19, 22)}


def _states(N, uniform):
    """Point states (B of them); uniform: all at the displacement gradient G."""
    from oracle import cp_local
    rng = np.random.default_rng(3 + N)
    H, Fp, g, slip, q = random_states(B, N, rng, table=TABLE[N])
    R = cp_local.rot_mat_from_quat(q)
    xm = np.full(B, 0.02)
    if uniform:
        H = np.broadcast_to(G, (B, 3, 3)).copy()
    kind = np.arange(B) % 4
    R[kind == 1] = R[kind == 1].astype(np.float32).astype(float)
    R[kind == 2, 0, 1] += 1e-3
    xm[kind == 3] = 1.0
    return H, Fp, g, slip, R, xm


def _material(N):
    import cpfem_amd as C
    return C.Material(slip="fcc12" if N == 12 else "bcc24", layout="9", self_block=True, g0=88.0, **FCC_304)


def _oracle_material(N, xm):
    from oracle import cp_local
    k = {a: v for a, v in FCC_304.items() if a != "xm"}
    return cp_local.Material(cp_local.schmid_tensors(slip_table(TABLE[N])), xm=xm, self_block=True, **k)


def _params(states, idx):
    H, Fp, g, slip, R, xm = states
    per = lambda k: np.full(len(idx), FCC_304[k])  # noqa: E731
    return [Fp[idx], g[idx], slip[idx], R[idx], per("gss_a"), per("h"), per("t_sat"), xm[idx], per("r")]


def _problem(N, n):
    """Cube of n^3 elements whose points hold the repeated states; displacement of gradient G."""
    import cpfem_amd as C
    m = C.box_mesh(n, n, n, 1.0, 1.0, 1.0)
    prob = C.CrystalPlasticity(C.Mesh(m.points, m.cells_dict["hexahedron"]), dirichlet_bc_info=None,
                               additional_info=(np.array([[1.0, 0, 0, 0]]), np.zeros(n ** 3, dtype=np.int64)), material=_material(N))
    prob.dt = 0.5
    states = _states(N, True)
    idx = np.arange(8 * n ** 3) % B
    params = [torch.as_tensor(np.ascontiguousarray(p.reshape((n ** 3, 8) + p.shape[1:])), device="cuda") for p in _params(states, idx)]
    prob.set_params(params)
    dofs = torch.as_tensor((np.asarray(m.points) @ G.T).ravel(), device="cuda")
    return prob, params, dofs, states, idx


_references = {}


def _reference(N, uniform):
    from oracle import cp_local
    if (N, uniform) not in _references:
        H, Fp, g, slip, R, xm = states = _states(N, uniform)
        ref = cp_local.local_update(H, Fp, g, slip, R, _oracle_material(N, xm), 0.5)
        assert not ref["capped"].any()
        _references[N, uniform] = states, ref
    return _references[N, uniform]


def _rel(a, b):
    a, b = a.reshape(len(a), -1), b.reshape(len(b), -1)
    return np.linalg.norm(a - b, axis=1) / np.linalg.norm(b, axis=1)


@pytest.mark.parametrize("N, Q", [(12, 512), (12, 47616), (12, 48128), (12, 84992), (12, 86016), (24, 512), (24, 19968), (24, 20480),
                                  (24, 48128), (24, 86016)])
def test_stress_and_history_at_every_lane_count(N, Q):
    states, ref = _reference(N, False)
    prob = _problem(N, 2)[0]
    idx = np.arange(Q) % B
    tensor_map, update_map = prob.get_maps()
    H = torch.as_tensor(states[0][idx], device="cuda")
    iv = [torch.as_tensor(np.ascontiguousarray(p), device="cuda") for p in _params(states, idx)]
    P = tensor_map(H, *iv).cpu().numpy()
    Fn, gn, sn = (t.cpu().numpy() for t in update_map(H, *iv)[:3])
    for a in (P, Fn, gn, sn):  # the same point has the same bits everywhere in the batch
        np.testing.assert_array_equal(a.reshape((Q // B, B) + a.shape[1:]), np.broadcast_to(a[:B], (Q // B, B) + a.shape[1:]))
    errors = _rel(P[:B], ref["P"]), _rel(Fn[:B], ref["Fp_inv_new"]), _rel(gn[:B], ref["g_new"])
    print(N, Q, [f"{e.max():.1e}" for e in errors], flush=True)
    assert errors[0].max() < 1e-10
    assert errors[1].max() < 1e-12
    assert errors[2].max() < 1e-12
    np.testing.assert_allclose(sn[:B], ref["slip_new"], rtol=1e-9, atol=1e-15)


def _forces(prob, P):
    """Nodal forces of the points' stresses P (Q, 3, 3), in numpy."""
    sg, w = prob.fes[0].shape_grads, prob.fes[0].JxW
    cells = np.asarray(prob.fes[0].cells)
    fe = np.einsum("eqij,eqaj,eq->eai", P.reshape(len(cells), 8, 3, 3), sg, w, optimize=True)
    out = np.zeros((prob.fes[0].num_total_nodes, 3))
    np.add.at(out, cells.ravel(), fe.reshape(-1, 3))
    return out.ravel()


@pytest.mark.parametrize("N, n", [(N, n) for N in (12, 24) for n in CUBES[N]])
def test_assembly_at_every_lane_count(N, n):
    import cpfem_amd as C
    states, ref = _reference(N, True)
    prob, params, dofs, _, idx = _problem(N, n)
    iters = torch.zeros(len(idx), dtype=torch.int32, device="cuda")
    res, mat = prob.assemble(dofs, apply_bc=False, iters=iters)
    res2, _ = prob.assemble(dofs, want_matrix=False, apply_bc=False)
    assert torch.equal(res, res2)
    assert int(iters.min()) > 0
    expected = _forces(prob, ref["P"][idx])
    # a matrix-vector product, with the oracle's tangents
    v = np.random.default_rng(1).normal(size=prob.ctx.n_dofs)
    cells = np.asarray(prob.fes[0].cells)
    grad = np.einsum("eak,eqal->eqkl", v.reshape(-1, 3)[cells], prob.fes[0].shape_grads, optimize=True).reshape(-1, 9)
    dP = np.einsum("qmn,qn->qm", ref["A"].reshape(B, 9, 9)[idx], grad)
    product = _forces(prob, dP.reshape(-1, 3, 3))
    y = C.BlockEllMatrix(prob.ctx, mat).to_scipy() @ v
    errors = (np.linalg.norm(res.cpu().numpy() - expected) / np.linalg.norm(expected), np.linalg.norm(y - product) / np.linalg.norm(product))
    print(N, n, [f"{e:.1e}" for e in errors], flush=True)
    assert errors[0] < 1e-10
    assert errors[1] < 1e-10
    sig = prob._compute_avg_stress_raw(dofs.reshape(-1, 3), params).cpu().numpy()
    avg = ref["sigma"][idx].reshape(-1, 8, 3, 3).mean(axis=1)
    assert _rel(sig, avg).max() < 1e-10


@pytest.mark.parametrize("N, n", [(N, n) for N in (12, 24) for n in CUBES[N]])
def test_point_vjp_at_every_lane_count(N, n):
    from cpfem_amd.adjoint import local_vjp
    from oracle import ad, cp_local
    prob, params, dofs, states, idx = _problem(N, n)
    rng = np.random.default_rng(9)
    Pb, Fb, gb, sb = (rng.normal(size=(B,) + s) for s in ((9,), (9,), (N,), (N,)))
    cell = rng.normal(size=(B // 8, 9))
    soa = lambda a: torch.as_tensor(np.ascontiguousarray(a.T), device="cuda")  # noqa: E731
    out = local_vjp(prob, dofs, params, Pbar=soa(Pb[idx]), sbar_cell=soa(cell[(np.arange(n ** 3)) % (B // 8)]), Fbar=soa(1e3 * Fb[idx]),
                    gbar=soa(gb[idx]), slipbar=soa(1e3 * sb[idx]))
    got = {k: v.t().cpu().numpy() for k, v in out.items()}
    if (N, "vjp") not in _references:
        H, Fp, g, slip, R, xm = states
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a)).requires_grad_(True)  # noqa: E731
        mat8 = np.stack([xm] + [np.full(B, FCC_304[k]) for k in ("gss_a", "h", "t_sat", "r", "C11", "C12", "C44")], axis=1)
        x = [t(a) for a in (H, Fp, g, R, mat8)]
        consts = ad.Consts(cp_local.schmid_tensors(slip_table(TABLE[N])), self_block=True)
        o = ad.point_outputs(x[0], x[1], x[2], torch.as_tensor(slip), x[3], x[4], consts, 0.5)
        spread = torch.as_tensor(np.repeat(cell, 8, axis=0)) / 8.0
        loss = ((o["P"].reshape(B, 9) * torch.as_tensor(Pb)).sum() + (o["sigma"].reshape(B, 9) * spread).sum()
                + 1e3 * (o["Fp_inv_new"].reshape(B, 9) * torch.as_tensor(Fb)).sum() + (o["g_new"] * torch.as_tensor(gb)).sum()
                + 1e3 * (o["slip_new"] * torch.as_tensor(sb)).sum())
        grads = torch.autograd.grad(loss, x)
        _references[N, "vjp"] = [a.numpy().reshape(B, -1) for a in grads]
    want = dict(zip(("Hbar", "Fpibar", "gbar_old", "Rbar", "pbar"), _references[N, "vjp"]))
    for k, w in want.items():
        scale = np.abs(w).max(axis=0)  # of each component over the points
        err = (np.abs(got[k] - w[idx]) / scale).max()
        print(N, n, k, f"{err:.1e}", flush=True)
        assert err < 5e-8


@pytest.mark.parametrize("N", [12, 24])
def test_tangents_of_a_batch(N):
    """Point updates with their tangents, of either form, among them unstrained points (converged before the first
    iteration) and one whose resistance is not a number, which does not reach its neighbours."""
    from cpfem_amd.models import local_full
    from oracle import cp_local
    H, Fp, g, slip, R, xm = (a.copy() for a in _states(N, False))
    H[64:96] = 0.0
    Fp[64:96] = np.eye(3)
    xm[64:96] = 0.02  # (at m = 1 the rate has a slope at zero stress; |x| is given none by the oracle)
    ref = cp_local.local_update(H, Fp, g, slip, R, _oracle_material(N, xm), 0.5)
    bad = 77
    g[bad, 5] = np.nan
    prob = _problem(N, 2)[0]
    out = local_full(prob, H, _params((H, Fp, g, slip, R, xm), np.arange(B)))
    rest = np.delete(np.arange(B), bad)
    strained = np.setdiff1d(rest, np.arange(64, 96))
    assert np.isnan(out["P"][bad]).any() and np.isfinite(out["A"][rest]).all()
    assert np.all(out["iters"][strained] > 0) and np.all(out["iters"][np.setdiff1d(np.arange(64, 96), [bad])] == 0)
    assert _rel(out["A"][rest], ref["A"].reshape(B, 9, 9)[rest]).max() < 1e-10
    assert _rel(out["P"][strained], ref["P"][strained]).max() < 1e-10
    assert np.abs(out["P"][np.setdiff1d(np.arange(64, 96), [bad])]).max() == 0.0
    assert _rel(out["Fp_inv_new"][rest], ref["Fp_inv_new"][rest]).max() < 1e-12
    assert _rel(out["g_new"][rest], ref["g_new"][rest]).max() < 1e-12
    np.testing.assert_allclose(out["slip_new"][rest], ref["slip_new"][rest], rtol=1e-9, atol=1e-15)


def test_parking_of_a_batch_with_one_lane_a_point():
    """Parking changes the time only, at the batch size it is made for (85,184 points, one lane each), with
    points of either form in every wave."""
    from cpfem_amd import configs
    w = configs.config5(n=22)
    prob = configs.build_problem(w)
    p0 = [p.clone() for p in prob.internal_vars]
    R = p0[3].reshape(-1, 3, 3)
    R[::3] = R[::3].float().double()
    p0[3] = R.reshape(p0[3].shape)
    sol0 = [torch.zeros(prob.fes[0].num_total_nodes, 3, dtype=torch.float64, device="cuda")]
    _, sol, _ = configs.run_steps(prob, w, p0, sol0, 0, 1, {"precision": "fp64"})
    prob.set_params(p0)
    dofs = sol[0].reshape(-1).clone()
    out = {}
    for lanes in (0, 8, 63):
        prob.ctx.set_point_park(lanes)
        prob.ctx.point_counts(reset=True)
        it = torch.empty(w.n_qp, dtype=torch.int32, device="cuda")
        res, mat = prob.assemble(dofs, iters=it)
        out[lanes] = res, mat.clone(), it, prob.ctx.point_counts(reset=True)
    prob.ctx.set_point_park(0)
    assert out[0][3][2] == 0 and out[0][2].max() > out[0][2].min()
    for lanes in (8, 63):
        for a, b in zip(out[lanes][:3], out[0][:3]):
            assert torch.equal(a, b)
        assert out[lanes][3][0] == out[0][3][0]  # the same total of Newton iterations
        assert out[lanes][3][2] > 0
