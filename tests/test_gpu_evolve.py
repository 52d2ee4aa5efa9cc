"""Time evolution with the expansion's terms added in the recursion steps: one to
about forty terms (every remainder of three), one and many states (both widths'
kernels), dictionary and plain operators, rows at a block's edges, against the
oracle at the tolerance of the time correlations (1e-10 of the largest)."""
import numpy as np
import pytest

import linqt_amd as lq
from conftest import random_upper_csr
from linqt_amd import lattices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [0.0, 1e-6, 1e-4, 1e-3, 4e-3, 0.02, 0.05, 0.2, 2.0])
@pytest.mark.parametrize("form,R", [("dict", 1), ("dict", 5), ("plain", 2), ("plain", 33)])
def test_evolution_terms(ctx, oracle, form, R, dt):
    print("[case] evolve", form, R, dt, flush=True)
    if form == "dict":
        m = lattices.square_anderson(9, W=0.0, seed=1)
        n, args, a = m.n, (m.rowptr, m.col, m.val), 4.6
    else:
        n, a = 257, 8.0
        args = random_upper_csr(n, 3.0 / n, 8, diag=True)
    G = lq.SparseMatrix(ctx, n, *args).Rescale(1 / a, 0.0)
    O = oracle.Op(n, *args).rescale(1 / a, 0.0)
    phi = lattices.random_phase_states(n, R, seed=R)
    got = lq.time_correlations(G, None, None, phi, 6, 3, dt, 2 * a, 0.1)
    ref = oracle.time_correlations(O, None, None, phi, 6, 3, dt, 2 * a, 0.1)
    assert np.abs(got - ref).max() <= 1e-10 * np.abs(ref).max()
