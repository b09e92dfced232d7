"""The multigrid solve at box shapes whose last level lies at the edges of the dense inverse: of exactly 768
rows (twelve full tiles; reached with even and with odd counts), 756, 864 (one level more, then 240 rows in
four tiles) and 192 rows (three full tiles) below a level of 1029.  Bars of test_gpu_multigrid."""
import pytest

from test_gpu_multigrid import OPTS, _check, _system

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.mark.parametrize("n", [(6, 14, 14), (5, 13, 13), (10, 10, 12), (10, 10, 13), (12, 12, 12)])
def test_last_levels_at_the_edges_of_the_dense_inverse(n):
    prob, mat, b, x0 = _system(n)
    for precision in ("fp64", "mixed"):
        _, k = _check(prob, mat, b, x0, dict(OPTS, precision=precision))
        assert 0 < k <= 30
