"""The overlap solver's restart and its queue of iterations.

S upper bidiagonal (1, 0.3) and a right-hand side along the last unit vector: after
one iteration the residual is exactly orthogonal to the first one, and the solver
has to start anew from the x it has, within iterations that are queued already."""
import numpy as np
import pytest

import linqt_amd as lq
from linqt_amd import io

pytestmark = pytest.mark.gpu


def _bidiagonal(n):
    rp = np.append(np.arange(0, 2 * n, 2), 2 * n - 1).astype(np.int32)
    cl = np.array([c for i in range(n) for c in (i, i + 1)][: 2 * n - 1], np.int32)
    v = np.where(np.arange(2 * n - 1) % 2, 0.3, 1.0).astype(complex)
    return io.CSR(n, rp, cl, v)


@pytest.mark.parametrize("n", [40, 300])
def test_restart(ctx, oracle, n):
    print("[case] restart", n, flush=True)
    S = _bidiagonal(n)
    Sg = lq.SparseMatrix(ctx, n, S.rowptr, S.col, S.val, fill=lq.LQ_FILL_GENERAL)
    b = np.zeros(n, complex)
    b[-1] = 2.0
    for maxit in (1, 2, 3, 4, 2000):
        x, it, err = lq.overlap_solve(Sg, b, tol=1e-13, maxit=maxit)
        xo, ito, erro = oracle.overlap_solve(S, b, tol=1e-13, maxit=maxit)
        assert it == ito if maxit < 2000 else abs(it - ito) <= 1 and err <= 1e-13
        assert np.abs(x - xo).max() <= 1e-11 * np.abs(xo).max()


def test_restart_in_a_long_queue(ctx, oracle):
    """H keeps only the last element of a vector: the first solve takes many
    iterations, the ones after it break down in the first of those queued."""
    print("[case] restart in a queue", flush=True)
    n = 40
    S = _bidiagonal(n)
    Sg = lq.SparseMatrix(ctx, n, S.rowptr, S.col, S.val, fill=lq.LQ_FILL_GENERAL)
    rp = np.zeros(n + 1, np.int32)
    rp[-1] = 1
    one = (rp, np.array([n - 1], np.int32), np.array([0.75 + 0j]))
    H, Ho = lq.SparseMatrix(ctx, n, *one), oracle.Op(n, *one)
    phi = np.random.default_rng(4).normal(size=(1, n)) + 0j
    mu = lq.spectral_moments_nonorth(H, None, Sg, phi, 5, tol=1e-13)
    ref = oracle.spectral_moments_nonorth(Ho, None, S, phi, 5, tol=1e-13)
    assert np.abs(mu - ref).max() <= 1e-10 * np.abs(ref).max()


def test_queue_is_bounded(ctx):
    """A solve of many iterations, then one of none: the second may queue no more
    than 16 iterations of two products each past its end, and so may the first."""
    print("[case] queue bound", flush=True)
    n = 400
    rows, cols, vals = [], [], []
    for i in range(n):
        for c, v in ((i - 1, -1.0), (i, 2.001), (i + 1, -1.0)):
            if 0 <= c < n:
                rows.append(i), cols.append(c), vals.append(v)
    rp = np.append(0, np.cumsum(np.bincount(rows, minlength=n))).astype(np.int32)
    Sg = lq.SparseMatrix(ctx, n, rp, np.array(cols, np.int32), np.array(vals, complex), fill=lq.LQ_FILL_GENERAL)
    H = lq.SparseMatrix(ctx, n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.zeros(n, complex))
    phi = np.random.default_rng(3).normal(size=(1, n)) + 0j
    info = {}
    ctx.set_timing(True)
    ctx.reset_timing()
    try:
        lq.spectral_moments_nonorth(H, None, Sg, phi, 2, tol=1e-10, info=info)
        launches = ctx.timing()["spmv_launches"]
    finally:
        ctx.set_timing(False)
    its = info["iterations"]
    assert its > 80
    assert 2 * its <= launches <= 2 * its + 2 * 2 * 16 + 2 + 2  # a restart's product; H's two
