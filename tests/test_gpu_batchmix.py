"""Jobs of every padded vector width in one launch, of one row to several blocks,
with dictionary and plain operators and equal and unequal slices (both kernels),
against the single-job solver, bit for bit."""
import numpy as np
import pytest

import linqt_amd as lq
from conftest import random_upper_csr
from linqt_amd import lattices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unroll", [None, "4", "16"])
def test_widths_in_one_launch(ctx, monkeypatch, unroll):
    print("[case] batch widths", unroll, flush=True)
    if unroll:
        monkeypatch.setenv("LQ_BATCH_UNROLL", unroll)
    batch = lq.Batch(ctx)
    jobs = []
    for i, R in enumerate([1, 2, 3, 5, 9, 16, 17, 33, 64]):
        for n in (1, 65, 700 + i):
            rp, cl, v = random_upper_csr(n, min(0.5, 3.0 / n), n + R, diag=True)
            if i % 2:
                v = np.sign(v.real) + 0j  # few values: dictionary form
                v[cl == np.repeat(np.arange(n), np.diff(rp))] = 0.25
            jobs.append((lq.SparseMatrix(ctx, n, rp, cl, v).Rescale(1 / 12.0, 0.0), n, R, 40 + 7 * i))
        m = lattices.square_anderson(20 + i, W=0.5 * (i % 2), seed=i)
        jobs.append((lq.SparseMatrix.from_csr(ctx, m).Rescale(1 / 4.6, 0.0), m.n, R, 33))
    for _ in range(2):
        phis = [lattices.random_phase_states(n, R, seed=k) for k, (_, n, R, _) in enumerate(jobs)]
        ids = [batch.submit(H, phi, M) for (H, _, _, M), phi in zip(jobs, phis)]
        batch.run()
        for k, ((H, n, R, M), phi) in enumerate(zip(jobs, phis)):
            print("[job]", k, n, R, M, flush=True)
            assert np.array_equal(batch.result(ids[k]), lq.spectral_moments(H, None, phi, M))
