"""Kubo energy sums from transforms of the stored vectors against the oracle's
per-site DFT route, at the edges of the frequency sets (M = 256, 512, 768), with
one to three operators, ragged numbers of stored elements, several groups of
states and sections.

Tolerance 1e-10 of the largest value, as for every Kubo sum: both sides round
each of the O(M) terms of a site to 1e-16 of its size and the oracle's angles
m theta to m 1e-16, which leaves about M 1e-16 <= 1e-13.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_inf
import linqt_amd as lq
from linqt_amd import lattices

pytestmark = pytest.mark.gpu


def _ops(ctx, oracle, L):
    H, Vx, Vy = lattices.haldane_honeycomb(L, seed=11)
    G = [lq.SparseMatrix.from_csr(ctx, m) for m in (H, Vx, Vy)]
    O = [oracle.Op.from_csr(m) for m in (H, Vx, Vy)]
    G[0].Rescale(1 / 4.6, 0.0)
    O[0].rescale(1 / 4.6, 0.0)
    return H.n, G, O


@pytest.mark.parametrize("formula,M,nump,L,R,nopr,ns", [
    (1, 129, 130, 3, 1, 1, 1), (0, 129, 258, 3, 3, 2, 1), (1, 255, 255, 4, 1, 2, 1), (1, 256, 300, 3, 1, 3, 1),
    (0, 257, 514, 3, 1, 1, 1), (1, 300, 301, 5, 1, 2, 5), (1, 512, 512, 3, 2, 2, 1), (0, 512, 1024, 3, 1, 3, 1),
    (1, 513, 513, 3, 1, 2, 1), (1, 641, 700, 3, 1, 1, 1), (0, 768, 768, 3, 1, 2, 1), (1, 769, 800, 3, 1, 1, 1),
    (1, 1030, 1030, 3, 1, 1, 1), (1, 200, 200, 3, 33, 2, 1), (1, 513, 513, 3, 2, 1, 1), (0, 640, 640, 4, 1, 1, 1)])
def test_kubo_sums_vs_oracle(ctx, oracle, formula, M, nump, L, R, nopr, ns):
    print("[case] kubo sums", formula, M, nump, L, R, nopr, ns, flush=True)
    n, G, O = _ops(ctx, oracle, L)
    phi = lattices.random_phase_states(n, R, seed=7)
    gops, oops = [G[1], G[2], None][:nopr], [O[1], O[2], None][:nopr]
    got = lq.kubo_fft(G[0], G[1], gops, phi, M, nump, formula, num_sections=ns)
    for o in range(nopr):
        ref, _ = oracle.kubo_fft(O[0], O[1], oops[o], phi, M, nump, formula, num_sections=ns)
        assert rel_inf(got[o], ref) < 1e-10, o


def test_no_table_is_allocated(oracle):
    """The sums take the place of the moment tables, so a solve of two operators at
    2048 orders and few elements stays below the tables' 134 MB of device memory."""
    print("[case] memory of the sums", flush=True)
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    c = lq.Context(0)
    n, G, _ = _ops(c, oracle, 3)
    phi = lattices.random_phase_states(n, 1, seed=7)
    lq.kubo_fft(G[0], G[1], [G[1], G[2]], phi, 200, 2048, 1)  # the device's own first allocations
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    before = free.value
    lq.kubo_fft(G[0], G[1], [G[1], G[2]], phi, 2048, 2048, 1)
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    assert before - free.value < 2 * 2048 * 2048 * 16
    c.close()
