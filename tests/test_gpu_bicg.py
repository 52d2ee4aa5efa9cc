"""The overlap solver with its scalars on the device, at the sizes of a block's
edges, against the oracle: stopped after few iterations (the rounding of a few
products and sums, 1e-11 of the largest element) and converged, in an order of
solves in which the queued iterations are too many, too few and right."""
import numpy as np
import pytest

import linqt_amd as lq
from conftest import random_upper_csr
from linqt_amd import io

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 64, 65, 255, 257, 5003])
def test_overlap_solve_edges(ctx, oracle, n):
    print("[case] overlap solve", n, flush=True)
    rp, cl, v = random_upper_csr(n, min(0.5, 4.0 / n), n, diag=True)
    rows = np.repeat(np.arange(n), np.diff(rp))
    v = 0.1 * v
    v[cl == rows] += 1.0
    S = io.CSR(n, rp, cl, v)
    Sg = lq.SparseMatrix(ctx, n, rp, cl, v, fill=lq.LQ_FILL_GENERAL)
    rng = np.random.default_rng(n)
    b = rng.normal(size=n) + 1j * rng.normal(size=n)
    for tol, maxit in ((1e-2, 2000), (1e-13, 2000), (1e-2, 2000), (1e-13, 1), (1e-13, 2), (1e-13, 2000), (1e-13, 2000)):
        x, it, err = lq.overlap_solve(Sg, b, tol=tol, maxit=maxit)
        xo, ito, erro = oracle.overlap_solve(S, b, tol=tol, maxit=maxit)
        assert it <= maxit and abs(it - ito) <= 1
        if maxit == 2000:  # both residuals within tol; S = 1 + 0.1 X, so |S^-1| < 2
            assert err <= tol and np.linalg.norm(x - xo) <= 4 * tol * np.linalg.norm(b)
        elif n > 2:
            assert it == ito == maxit
        if it == ito or tol == 1e-13 and maxit == 2000:
            assert np.abs(x - xo).max() <= 1e-11 * np.abs(xo).max()
