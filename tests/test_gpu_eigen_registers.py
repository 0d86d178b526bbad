"""The cooperative tridiagonalisation with a worker's columns in registers at
the edges of its shapes (64 rows a register, up to 3, 4 and 5 columns a wave,
640 rows in all) and just past them, against LAPACK: random matrices, and ones
that fall apart into blocks (zero reflectors)."""
import numpy as np
import pytest

from test_gpu_subspace import _check_pairs, _coop

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,workers", [(3, 1), (64, 8), (65, 8), (127, 12), (128, -1), (129, -1), (192, -1), (193, -1),
                                       (256, -1), (257, -1), (319, -1), (320, 20), (384, -1), (385, -1), (512, -1),
                                       (513, -1), (640, -1), (641, -1)])
def test_eigen_register_tridiagonalisation(m, workers):
    old = _coop([workers, 3, 1025, 1 << 21])
    try:
        rng = np.random.default_rng(m)
        B = rng.standard_normal((m, m))
        A = 0.5 * (B + B.T)
        _check_pairs(A, min(m, 40), f"registers x{workers} random")
        A[: m // 3, m // 3:] = 0.0
        A[m // 3:, : m // 3] = 0.0
        A[-1, :-1] = A[:-1, -1] = 0.0
        _check_pairs(A, min(m, 40), f"registers x{workers} blocks")
    finally:
        _coop(old)
