"""GPU parity tests of POTRI for orders up to 32 (four matrices per wavefront,
kb_inv.hip) against the oracle: the orders at the edges of its one- and
two-slot forms, batches that leave part of a wavefront empty, pointer arrays
with padded columns, a zero on the diagonal in either slot.

Bar: within 16 n eps of the oracle's inverse (max-norm, relative to its own);
the strict upper triangle and the padding (NaN) are not touched; a matrix with
a zero pivot keeps its bits and reports its index."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 18, 31, 32])
@pytest.mark.parametrize("batch", [1, 3, 4, 9])
def test_potri_small(p, n, batch):
    dt, eps = (np.float64, kt.EPS64) if p == "D" else (np.float32, kt.EPS32)
    pad, bad = 3, batch // 2
    A = po.gen_spd_shift_batch(50 + n, n, batch)
    Ls, buf = [], np.full((batch, n, n + pad), np.nan, dt)
    for b in range(batch):
        L = np.tril(po.potrf(po.col(A, b))[0]).astype(dt).astype(np.float64)
        if b == bad:
            L[n - 1, n - 1] = 0.0
            if n > 3:
                L[n // 2, n // 2] = 0.0
        Ls.append(L)
        for c in range(n):
            buf[b, c, c:n] = L[c:, c]
    d = kt.to_dev(buf)
    info = kt.to_dev(np.full(batch, -7, np.int32))
    h = kt.handle()
    ptrs = kt.ptr_array(d, batch, n * (n + pad))
    st = getattr(h.lib, "kblas%spotri_batch" % p)(h.h, b"L", n, kt.P(ptrs), n + pad, batch, kt.P(info))
    assert st == pykblas.KBLAS_Success
    got, inf = kt.to_host(d), kt.to_host(info)
    h.close()
    up = np.triu_indices(n, 1)
    for b in range(batch):
        X = got[b, :, :n].T
        assert np.all(np.isnan(X[up])) and np.all(np.isnan(got[b, :, n:]))
        if b == bad:
            assert inf[b] == (n // 2 + 1 if n > 3 else n)
            assert np.array_equal(got[b], buf[b], equal_nan=True)
            continue
        assert inf[b] == 0
        want = np.tril(po.potri(Ls[b])[0])
        assert np.max(np.abs(np.tril(X) - want)) <= 16 * n * eps * np.max(np.abs(want)), b
