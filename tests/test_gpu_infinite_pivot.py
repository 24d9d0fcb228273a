"""GPU test of FP32 POSV above order 64 with an infinity on A's diagonal at the
first column of a 16 x 16 diagonal tile: its column of L is zero below it, the
factorization goes on (info = 0), and the unknowns after it are those of the
system without that row and column.

Bar: info = 0; those unknowns within 64 n eps of the oracle's solution of the
smaller system (max-norm, relative to max(|X|, 1))."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(65, 32), (97, 48), (224, 112)])
@pytest.mark.parametrize("batch", [3, 1100])
def test_infinite_pivot(n, k, batch):
    torch = kt.torch_dev()
    nrhs = 5
    A = po.gen_spd_shift_batch(63, n, 1).astype(np.float32)
    B = po.gen_rhs_batch(73, n, nrhs, 1).astype(np.float32)
    keep = np.arange(n) != k
    Xk = po.posv("L", A[0][np.ix_(keep, keep)].T.astype(np.float64), B[0][:, keep].T.astype(np.float64))[1]
    A[0][k, k] = np.inf
    idx = torch.zeros(batch, dtype=torch.long, device="cuda")
    dA, dB = kt.to_dev(A)[idx], kt.to_dev(B)[idx]
    info = torch.full((batch,), -7, dtype=torch.int32, device="cuda")
    h = kt.handle()
    st = h.lib.kblasSposv_batch_strided(h.h, b"L", b"L", n, nrhs, kt.P(dA), n, n * n, kt.P(dB), n, n * nrhs, batch,
                                        kt.P(info))
    assert st == pykblas.KBLAS_Success
    assert int((info != 0).sum()) == 0
    X = kt.to_host(dB[-1]).T.astype(np.float64)
    h.close()
    assert np.max(np.abs(X[k + 1:] - Xk[k:])) <= 64 * n * kt.EPS32 * max(np.max(np.abs(Xk)), 1)
