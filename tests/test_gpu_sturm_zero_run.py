"""Sturm counts at a point that is exactly a run of equal, decoupled diagonal
entries: the leading minors there alternate between zero and powers of the
floor on e^2, and their scale must not be taken from the zero. The matrix is
diagonal (the reduction leaves it as it is), its first 16 rows the run, 40
slightly smaller entries behind them; the run's value is one of the 64 points
of the first multisection step, computed as the kernel does (with and without
a fused multiply-add, as it may be compiled)."""
from fractions import Fraction

import numpy as np
import pytest

from test_gpu_subspace import _eigen_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("point", [30, 36, 41, 50])
@pytest.mark.parametrize("fused", [True, False])
def test_counts_past_a_run_of_zero_minors(point, fused):
    run, small, norm = 16, 40, 0.9  # norm in [0.5, 1): no rescaling of the matrix
    m = run + small + 2
    pad = 2.1 * norm * 2.0 ** -52 * m
    lo = -norm - pad
    width, part = (norm + pad) - lo, point / 65.0
    c = float(Fraction(width) * Fraction(part) + Fraction(lo)) if fused else width * part + lo
    d = np.concatenate([np.full(run, c), c - 0.01 - 1e-4 * np.arange(small), [-norm, norm]])
    values, _ = _eigen_dev(np.diag(d), small + 1)
    # The bracket ends within a few ulps of the norm.
    assert np.abs(values - np.sort(d)[:small + 1]).max() < 1e-14
