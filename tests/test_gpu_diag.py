"""Energy-grid sums through a table's diagonals: the linear-grid tools on both
sides of the size from which they are used (64 x 64 moments), square and not,
and the Kubo sums of small tables (up to 128 orders), against the oracle.
Tolerance 1e-9 of the largest value, as for every energy grid.  Kind 5 (Sea)
prints a running sum that begins with the NaN of x = -1: only its energies and
the NaN can be compared."""
import numpy as np
import pytest

from conftest import rel_inf
import linqt_amd as lq
from linqt_amd import lattices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [1, 2, 3, 5, 6])
@pytest.mark.parametrize("M0,M1,nd", [(63, 65, 200), (64, 64, 2049), (65, 64, 65), (1, 4096, 40), (300, 17, 99),
                                      (129, 200, 2100)])
def test_linear_grid_by_diagonals(ctx, oracle, kind, M0, M1, nd):
    print("[case] linear grid", kind, M0, M1, nd, flush=True)
    rng = np.random.default_rng(M0 + 7 * M1)
    g = lambda M: (1.0 - np.arange(M) / M) ** 2  # noqa: E731
    mu = (rng.normal(size=(M0, M1)) + 1j * rng.normal(size=(M0, M1))) * np.outer(g(M0), g(M1))
    E, v = lq.linear_grid(ctx, kind, mu, 5000, 9.2, 0.3, nd)
    Eo, vo = oracle.linear_grid(kind, mu, 5000, 9.2, 0.3, nd)
    assert np.allclose(E, Eo, rtol=0, atol=1e-13)
    assert np.array_equal(np.isnan(v), np.isnan(vo)) and np.array_equal(np.isinf(v), np.isinf(vo))
    fin = np.isfinite(vo)
    assert fin.sum() == 0 if kind == 5 else fin.sum() >= len(vo) - 2
    if fin.any():
        assert rel_inf(v[fin], vo[fin]) < 1e-9


@pytest.mark.parametrize("formula,M,nump", [(1, 1, 3), (0, 2, 2), (1, 33, 40), (0, 65, 65), (1, 128, 129)])
def test_kubo_table_by_diagonals(ctx, oracle, formula, M, nump):
    print("[case] kubo table", formula, M, nump, flush=True)
    H, Vx, Vy = lattices.haldane_honeycomb(4, seed=5)
    G = [lq.SparseMatrix.from_csr(ctx, m) for m in (H, Vx, Vy)]
    O = [oracle.Op.from_csr(m) for m in (H, Vx, Vy)]
    G[0].Rescale(1 / 4.6, 0.0)
    O[0].rescale(1 / 4.6, 0.0)
    phi = lattices.random_phase_states(H.n, 2, seed=3)
    got = lq.kubo_fft(G[0], G[1], [G[1], G[2]], phi, M, nump, formula)
    for o, opr in enumerate(O[1:]):
        ref, _ = oracle.kubo_fft(O[0], O[1], opr, phi, M, nump, formula)
        assert rel_inf(got[o], ref) < 1e-10, o
