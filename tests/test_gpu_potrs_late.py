"""GPU test of POTRS of order 32 with one right-hand side on both sides of the
batch size where the kernel loads it after the factor instead of with it.

Bar: bit for bit the solutions of the same systems in a batch of nine, which are
within 16 n eps of the oracle's (max-norm, relative to max(|X|, 1))."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("side", ["L", "R"])
def test_potrs_one_rhs(p, side):
    torch = kt.torch_dev()
    dt, eps = (np.float64, kt.EPS64) if p == "D" else (np.float32, kt.EPS32)
    n, few = 32, 9
    A = po.gen_spd_shift_batch(280, n, few)
    Ls = np.array([np.tril(po.potrf(po.col(A, i))[0]).T for i in range(few)]).astype(dt)
    rows, cols = (n, 1) if side == "L" else (1, n)
    B = po.gen_rhs_batch(281, rows, cols, few).astype(dt)
    dL, dB = kt.to_dev(Ls), kt.to_dev(B)
    h = kt.handle()
    out = []
    for batch in (few, 8191, 8192, 8195):
        idx = torch.arange(batch, device="cuda") % few
        a, b = dL[idx], dB[idx]
        st = getattr(h.lib, "kblas%spotrs_batch_strided" % p)(h.h, side.encode(), b"L", rows, cols, kt.P(a), n, n * n,
                                                              kt.P(b), rows, n, batch)
        assert st == pykblas.KBLAS_Success
        out.append((idx, b))
    want = out[0][1]
    for idx, b in out[1:]:
        assert torch.equal(want[idx], b)
    X = kt.to_host(want)
    h.close()
    for i in range(few):
        Xo = po.potrs(side, Ls[i].T, B[i].T)
        assert np.max(np.abs(X[i].T - Xo)) <= 16 * n * eps * max(np.max(np.abs(Xo)), 1), i
