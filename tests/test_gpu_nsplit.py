"""The split of a contraction's K into chunks and the reduction of the partial
tables, at K below, at and just past the smallest chunks, for tables of one and of
several tiles, against numpy.  Tolerance 1e-13 of the product of the row norms'
maximum, as for every contraction."""
import ctypes as C

import numpy as np
import pytest

import linqt_amd as lq
from linqt_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ML,MR", [(1, 1), (5, 70), (100, 100), (128, 128), (129, 300), (260, 140)])
@pytest.mark.parametrize("K", [1, 17, 63, 64, 65, 511, 512, 1000, 8191, 20011])
def test_mom_table_split(ctx, ML, MR, K):
    print("[case] split", ML, MR, K, flush=True)
    rng = np.random.default_rng(ML + 3 * MR + 7 * K)
    ld = K + 3
    L = rng.normal(size=(ML, ld)) + 1j * rng.normal(size=(ML, ld))
    R = rng.normal(size=(MR, ld)) + 1j * rng.normal(size=(MR, ld))
    out = np.zeros((ML, MR), complex)
    dp = C.POINTER(C.c_double)
    p = [ctx.alloc(a.nbytes) for a in (L, R, out)]
    try:
        ctx.upload(p[0], L)
        ctx.upload(p[1], R)
        _lib.call("lq_compute_mom_table", ctx.h, C.cast(p[0], dp), C.c_longlong(ld), ML, C.cast(p[1], dp),
                  C.c_longlong(ld), MR, C.c_longlong(K), C.cast(p[2], dp), MR)
        ctx.download(p[2], out)
    finally:
        for q in p:
            ctx.free(q)
    ref = L[:, :K].conj() @ R[:, :K].T
    scale = np.linalg.norm(L[:, :K], axis=1).max() * np.linalg.norm(R[:, :K], axis=1).max()
    assert np.abs(out - ref).max() < 1e-13 * scale
