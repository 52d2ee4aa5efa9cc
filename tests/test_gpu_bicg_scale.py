"""Overlap solves of scaled systems.  A power of two in front of the right-hand
side or of S scales every vector and scalar of BiCGSTAB by a power of two and
changes no rounding, so the solution is the unscaled one's times that power, bit
for bit, in the same number of iterations."""
import numpy as np
import pytest

import linqt_amd as lq
from conftest import random_upper_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eb,es", [(-332, 0), (-280, 0), (-256, 0), (256, 0), (332, 0), (0, -560), (0, 300)])
def test_scaled_systems(ctx, eb, es):
    print("[case] scaled overlap solve", eb, es, flush=True)
    n = 301
    rp, cl, v = random_upper_csr(n, 4.0 / n, 5, diag=True)
    rows = np.repeat(np.arange(n), np.diff(rp))
    v = 0.1 * v
    v[cl == rows] += 1.0 + 0.5j
    rng = np.random.default_rng(6)
    b = rng.normal(size=n) + 1j * rng.normal(size=n)
    plain = lq.SparseMatrix(ctx, n, rp, cl, v, fill=lq.LQ_FILL_GENERAL)
    x, it, err = lq.overlap_solve(plain, b, tol=1e-10)
    assert 2 < it < 100 and err <= 1e-10
    sb, ss = 2.0 ** eb, 2.0 ** es
    other = lq.SparseMatrix(ctx, n, rp, cl, ss * v, fill=lq.LQ_FILL_GENERAL)
    xs, its, errs = lq.overlap_solve(other, sb * b, tol=1e-10)
    assert its == it and errs == err
    assert np.array_equal(xs, x * (sb / ss))
