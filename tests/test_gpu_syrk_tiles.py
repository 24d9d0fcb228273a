"""GPU tests of SYRK at the work where it changes to 64 x 64 workgroup tiles: the
smallest batches that take them and the largest that do not (FP32 with k above 16:
1,536 tiles up to order 128, 640 above; FP64 above order 192 with k of 48 or more:
512 tiles).

Bar: 16 k eps of the largest element of the result, against NumPy in FP64; the
other triangle (NaN) is neither read nor written."""
import numpy as np
import pytest

import kbtest as kt
import pykblas

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("p,n,k,batch", [("S", 64, 17, 1535), ("S", 64, 17, 1536), ("S", 100, 33, 511), ("S", 100, 33, 512),
                                         ("S", 70, 16, 3), ("S", 161, 40, 106), ("S", 161, 40, 107),
                                         ("D", 225, 64, 51), ("D", 225, 48, 52), ("D", 225, 47, 52),
                                         ("D", 256, 100, 52)])
def test_syrk_tiles(trans, uplo, p, n, k, batch):
    dt, eps = (np.float64, kt.EPS64) if p == "D" else (np.float32, kt.EPS32)
    rng = np.random.default_rng(n + k + batch)
    few = 8   # the batch repeats these
    rows, cols = (n, k) if trans == "N" else (k, n)
    A = rng.standard_normal((few, cols, rows)).astype(dt)   # [matrix, column, row]
    C = rng.standard_normal((few, n, n)).astype(dt)
    low = np.tri(n, dtype=bool).T   # column-major: C[i, c, r] with r >= c
    keep = low if uplo == "L" else low.T
    C[:, ~keep] = np.nan
    idx = np.arange(batch) % few
    dA, dC = kt.to_dev(A[idx]), kt.to_dev(C[idx])
    h = kt.handle()
    st = getattr(h.lib, "kblas%ssyrk_batch_strided" % p)(h.h, uplo.encode(), trans.encode(), n, k, 0.5, kt.P(dA), rows,
                                                         rows * cols, -1.0, kt.P(dC), n, n * n, batch)
    assert st == pykblas.KBLAS_Success
    R = kt.to_host(dC)
    h.close()
    M = A.astype(np.float64).transpose(0, 2, 1)   # rows x cols
    M = M if trans == "N" else M.transpose(0, 2, 1)
    want = 0.5 * (M @ M.transpose(0, 2, 1)) - C   # (the product is symmetric)
    for b in range(batch):
        w = want[b % few]
        assert np.all(np.isnan(R[b][~keep])), b
        assert np.max(np.abs(R[b][keep] - w[keep])) <= 16 * k * eps * np.max(np.abs(w[keep])), b
