"""Pivots that nearly vanish where the direct solver's second front meets them, and not after the rows before
them are eliminated: one front from the near end solves such a system to full accuracy, and so has the call to.

The entry is the first diagonal one of the last tile of the band, in a stiffness matrix whose rows are
of the order of 1e5.  The bounds are those of the solver's other comparisons with scipy's sparse LU: 1e-9 without
refinement, 1e-11 after two steps."""
import numpy as np
import pytest

from test_gpu_band_tiles import _check, _system

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [(1, 1, 44), (6, 6, 6)])  # bands of nine and of seventeen tiles
@pytest.mark.parametrize("size", [1e-3, 1e-7, 1e-10, 1e-12, 1e-15, 1e-17, -1e-16])
def test_pivots_that_nearly_vanish_from_the_far_end(n, size):
    prob, mat, b = _system(*n)
    rows = len(b)
    row = (rows - 1) // 64 * 64
    node, comp = divmod(row, 3)
    slot = int(np.nonzero(prob.ctx.pattern()[1][:, node] == node)[0][0])
    entry = mat.view(-1, rows)[3 * slot + comp]
    assert float(entry[row]) > 1e4
    entry[row] *= size
    _check(prob, mat, b)


def test_a_zero_row_still_fails():
    from cpfem_amd.solver import direct_solve
    prob, mat, b = _system(1, 1, 44)
    mat.view(-1, len(b))[:, 512] = 0.0
    with pytest.raises(RuntimeError, match="pivot"):
        direct_solve(prob, mat, b, {"umfpack_solver": {}})
