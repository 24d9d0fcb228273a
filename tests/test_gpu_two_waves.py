"""GPU tests of POTRS above order 64 at the batch sizes where its kernel changes:
four waves per matrix, four waves with at most four matrices to a CU, two waves
per matrix (batches of more than 1,280 in FP64, 1,536 in FP32, for few right-hand
sides), more matrices than workgroups.

Bar: bit for bit the solutions of the same systems in a batch of seven, which are
within 64 n eps of the oracle's (max-norm, relative to max(|X|, 1))."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po

pytestmark = pytest.mark.gpu

FEW = 7


@pytest.fixture(scope="module")
def h():
    hh = kt.handle()
    yield hh
    hh.close()


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("side", ["L", "R"])
@pytest.mark.parametrize("n,nrhs", [(65, 1), (97, 24), (100, 25), (128, 9), (129, 8), (160, 16), (224, 4), (225, 32)])
def test_potrs_batches(h, p, side, n, nrhs):
    torch = kt.torch_dev()
    dt, eps = (np.float64, kt.EPS64) if p == "D" else (np.float32, kt.EPS32)
    A = po.gen_spd_shift_batch(260 + n, n, FEW)
    Ls = np.array([np.tril(po.potrf(po.col(A, i))[0]).T for i in range(FEW)]).astype(dt)
    rows, cols = (n, nrhs) if side == "L" else (nrhs, n)
    B = po.gen_rhs_batch(270 + nrhs, rows, cols, FEW).astype(dt)
    dL, dB = kt.to_dev(Ls), kt.to_dev(B)
    want = None
    for batch in (FEW, 1030, 1290, 1700, 2070, 4105):
        idx = torch.arange(batch, device="cuda") % FEW
        a, b = dL[idx], dB[idx]
        st = getattr(h.lib, "kblas%spotrs_batch_strided" % p)(h.h, side.encode(), b"L", rows, cols, kt.P(a), n, n * n,
                                                              kt.P(b), rows, rows * cols, batch)
        assert st == pykblas.KBLAS_Success
        if want is None:
            want = b
            X = kt.to_host(b)
            for i in range(FEW):
                Xo = po.potrs(side, np.asfortranarray(Ls[i].T.astype(np.float64)),
                              np.asfortranarray(B[i].T.astype(np.float64)))
                Xo = Xo[0] if isinstance(Xo, tuple) else Xo
                assert np.max(np.abs(X[i].T - Xo)) <= 64 * n * eps * max(np.max(np.abs(Xo)), 1), i
        else:
            assert torch.equal(want[idx], b), batch
