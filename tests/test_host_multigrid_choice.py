"""The choice between the multigrid and the Jacobi preconditioner (cpfem_multigrid_pays, host code of
libcpfem_hip.so; no device needed), on box meshes whose two solves were timed: it is multigrid's
where that was faster by more than a half, and Jacobi's where the multigrid attempt was the slower one.  The
same mesh in other units, turned or numbered along another axis gets the same answer."""
import ctypes
import os

import numpy as np
import pytest

pytest.importorskip("torch")

SYMMETRY, HELD = "symmetry planes, driven top", "bottom and top held"

# elements, their proportions, how the box is held, time of the Jacobi solve over that of the other
MEASURED = [
    ((24, 24, 24), (1, 1, 1), SYMMETRY, 3.4), ((24, 24, 24), (1, 1, 1), HELD, 2.4), ((48, 48, 48), (1, 1, 1), HELD, 7.3),
    ((16, 16, 16), (1, 1, 1), SYMMETRY, 2.6), ((7, 7, 7), (1, 1, 1), SYMMETRY, 1.8), ((8, 8, 8), (1, 1, 2), SYMMETRY, 1.7), ((8, 12, 20), (1, 1, 1), HELD, 2.6),
    ((40, 3, 3), (1, 1, 1), SYMMETRY, 2.0), ((24, 24, 6), (1, 1, 1), SYMMETRY, 2.6), ((100, 2, 2), (1, 1, 1), SYMMETRY, 3.2),
    ((24, 24, 24), (1, 1, 2), SYMMETRY, 2.9), ((24, 24, 24), (1, 1, 0.5), HELD, 1.6), ((24, 24, 24), (1, 1, 0.1), SYMMETRY, 2.5),
    ((24, 24, 24), (1, 1, 4), HELD, 3.7), ((24, 24, 24), (1, 2, 2), SYMMETRY, 3.0), ((48, 48, 48), (1, 5, 5), SYMMETRY, 4.6),
    ((16, 16, 16), (1, 1, 2), HELD, 2.5), ((24, 24, 24), (1, 1, 10), SYMMETRY, 0.9), ((24, 24, 24), (1, 1, 10), HELD, 0.89), ((24, 24, 24), (1, 1, 0.05), HELD, 0.33),
    ((24, 24, 24), (1, 1, 0.1), HELD, 0.47), ((24, 24, 24), (10, 1, 1), HELD, 0.61), ((24, 24, 24), (1, 10, 10), HELD, 0.95),
    ((24, 24, 24), (1, 3, 9), HELD, 0.87), ((16, 16, 16), (1, 1, 0.2), HELD, 0.57), ((16, 16, 16), (1, 1, 7), SYMMETRY, 0.76),
    ((16, 16, 16), (4, 2, 1), HELD, 0.81), ((8, 12, 20), (1, 1, 5), SYMMETRY, 0.86), ((24, 24, 6), (1, 1, 1), HELD, 0.48),
    ((24, 24, 6), (1, 1, 2), HELD, 0.43), ((32, 32, 4), (1, 1, 4), HELD, 0.61), ((32, 32, 4), (1, 1, 10), SYMMETRY, 0.44),
    ((24, 24, 8), (1, 1, 0.5), HELD, 0.62), ((24, 24, 7), (1, 1, 1), HELD, 0.88),
]


def _library():
    from cpfem_amd import _native as N
    if not os.path.exists(N.LIB_PATH):
        pytest.skip("libcpfem_hip.so not built")
    return N.load_library()


def _box(n, h):
    """Nodes (x fastest) and the indices of their coordinates."""
    z, y, x = np.meshgrid(*[np.arange(k + 1) for k in n[::-1]], indexing="ij")
    ijk = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    return ijk * np.asarray(h, dtype=float), ijk


def _held(n, ijk, how):
    at = lambda d, v: np.flatnonzero(ijk[:, d] == v)  # noqa: E731
    if how is HELD:
        sets = [(at(2, v), c) for v in (0, n[2]) for c in range(3)]
    else:
        sets = [(at(0, 0), 0), (at(1, 0), 1), (at(2, 0), 2), (at(2, n[2]), 2)]
    return np.concatenate([3 * nodes + c for nodes, c in sets]).astype(np.int64)


def _pays(L, n, points, dofs):
    dims = np.asarray([k + 1 for k in n], dtype=np.int64)
    points, dofs, out = np.ascontiguousarray(points), np.ascontiguousarray(dofs), ctypes.c_int32(-1)
    assert L.cpfem_multigrid_pays(dims.ctypes.data, points.ctypes.data, len(dofs), dofs.ctypes.data, ctypes.byref(out)) == 0
    return out.value


@pytest.mark.parametrize("n, h, how, gain", MEASURED)
def test_the_faster_solve_is_chosen(n, h, how, gain):
    L = _library()
    points, ijk = _box(n, h)
    dofs = _held(n, ijk, how)
    want = 1 if gain > 1.5 else 0
    assert _pays(L, n, points, dofs) == want
    assert _pays(L, n, 1e-3 * points, dofs) == want
    # the coordinates exchanged (the box lies along another axis, the numbering stays)
    assert _pays(L, n, points[:, [2, 0, 1]], 3 * (dofs // 3) + np.array([1, 2, 0])[dofs % 3]) == want
    # the box axes exchanged in the numbering
    turned = [n[1], n[2], n[0]]
    tp, tijk = _box(turned, [h[1], h[2], h[0]])
    old = (tijk[:, 2]) + (n[0] + 1) * (tijk[:, 0] + (n[1] + 1) * tijk[:, 1])  # old node of each new one
    new = np.empty(len(old), dtype=np.int64)
    new[old] = np.arange(len(old))
    assert _pays(L, turned, points[old], 3 * new[dofs // 3] + dofs % 3) == want


def test_the_most_stretched_element_decides():
    """A mesh graded towards a face, whose mean proportions alone would do."""
    L = _library()
    n = (24, 24, 24)
    points, ijk = _box(n, (1, 1, 1))
    assert _pays(L, n, points, _held(n, ijk, SYMMETRY)) == 1
    graded = points.copy()
    graded[:, 2] = 24 * (ijk[:, 2] / 24.0) ** 4
    assert _pays(L, n, graded, _held(n, ijk, SYMMETRY)) == 0


def test_a_box_that_is_not_held():
    L = _library()
    n = (24, 24, 24)
    points, _ = _box(n, (1, 1, 1))
    assert _pays(L, n, points, np.zeros(0, dtype=np.int64)) == 1


def test_bad_arguments_are_refused():
    L = _library()
    points, _ = _box((3, 3, 3), (1, 1, 1))
    dims, one, out = np.array([4, 4, 4], dtype=np.int64), np.array([3 * 64], dtype=np.int64), ctypes.c_int32(0)
    call = L.cpfem_multigrid_pays
    assert call(dims.ctypes.data, points.ctypes.data, 1, one.ctypes.data, ctypes.byref(out)) != 0
    assert call(dims.ctypes.data, points.ctypes.data, 1, None, ctypes.byref(out)) != 0
    dims[1] = 1
    assert call(dims.ctypes.data, points.ctypes.data, 0, None, ctypes.byref(out)) != 0
