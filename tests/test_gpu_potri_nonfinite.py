"""GPU tests of POTRI up to order 32 on factors with an infinity or a NaN below
the diagonal: an element L(k, j) that is not finite reaches the elements of
L^-1 at or below row k and at or left of column j, so of (L L^T)^-1 = L^-T L^-1
the elements whose row and column both lie right of column j stay finite
(LAPACK's dpotri as well).  The neighbours in the same wavefront keep their bits.

Bar: those elements within 16 n eps of the oracle's (max-norm of that block), the
rest of the lower triangle not finite where the product runs over the bad rows."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("n,k,j", [(2, 1, 0), (9, 5, 2), (16, 15, 0), (16, 8, 7), (20, 18, 3), (31, 17, 16), (32, 16, 15),
                                   (32, 31, 10)])
def test_potri_nonfinite(p, value, n, k, j):
    dt, eps = (np.float64, kt.EPS64) if p == "D" else (np.float32, kt.EPS32)
    batch, bad = 6, 2
    A = po.gen_spd_shift_batch(50 + n, n, batch)
    Ls = [np.tril(po.potrf(po.col(A, b))[0]).astype(dt).astype(np.float64) for b in range(batch)]
    h = kt.handle()
    res = []
    for v in (None, value):
        buf = np.array([L.T for L in Ls]).astype(dt)
        if v is not None:
            buf[bad, j, k] = v
        d = kt.to_dev(buf)
        info = kt.to_dev(np.full(batch, -7, np.int32))
        st = getattr(h.lib, "kblas%spotri_batch_strided" % p)(h.h, b"L", n, kt.P(d), n, n * n, batch, kt.P(info))
        assert st == pykblas.KBLAS_Success
        assert not kt.to_host(info).any()
        res.append(kt.to_host(d))
    h.close()
    for b in range(batch):
        if b != bad:
            assert np.array_equal(res[0][b], res[1][b]), b
    X = res[1][bad].T.astype(np.float64)
    want = np.tril(po.potri(Ls[bad])[0])[j + 1:, j + 1:]
    assert np.max(np.abs(np.tril(X[j + 1:, j + 1:]) - want)) <= 16 * n * eps * np.max(np.abs(want))
    assert not np.isfinite(X[j, j]) and not np.any(np.isfinite(X[k:, j]))
