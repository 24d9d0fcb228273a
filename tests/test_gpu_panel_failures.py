"""GPU tests of the Cholesky above order 64 on matrices that are not positive
definite, failing in the first, a middle and the last panel of 32 columns.

LAPACK's info; A from the failing panel's rows below its diagonal block on, the
right-hand sides' rows from the failing panel on, and all padding keep their
bits; the columns and right-hand-side rows of the panels before are those of a
factorization that does not fail.  Batches beyond the number of workgroups a
launch has (2,048) reuse a workgroup after a failed matrix: the others keep the
bits they have in a small batch, with two and with four waves per matrix."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po

pytestmark = pytest.mark.gpu

POSV = "kblas%sposv_batch_strided"


@pytest.fixture(scope="module")
def h():
    hh = kt.handle()
    yield hh
    hh.close()


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("side", ["L", "R"])
@pytest.mark.parametrize("n,nrhs", [(65, 3), (97, 17), (150, 5), (290, 33)])
def test_failing_panel(h, p, side, n, nrhs):
    dt = np.float64 if p == "D" else np.float32
    cols = sorted({0, 3, 31, 32, n // 2, (n - 1) // 32 * 32, n - 1})   # 0-based failing columns
    batch, pad = len(cols) + 1, 2
    A = po.gen_spd_shift_batch(61, n, 1)[0].astype(dt)
    rows, ncol = (n, nrhs) if side == "L" else (nrhs, n)
    B = po.gen_rhs_batch(71, rows, ncol, 1)[0].astype(dt)   # (column, row)
    a0 = np.full((batch, n, n + pad), np.nan, dt)
    a0[:, :, :n] = A
    b0 = np.full((batch, ncol, rows + pad), np.nan, dt)
    b0[:, :, :rows] = B
    for i, c in enumerate(cols):
        a0[i, c, c] = -1.0
    dA, dB, info = kt.to_dev(a0), kt.to_dev(b0), kt.to_dev(np.full(batch, -7, np.int32))
    st = getattr(h.lib, POSV % p)(h.h, side.encode(), b"L", rows, ncol, kt.P(dA), n + pad, n * (n + pad), kt.P(dB),
                                  rows + pad, ncol * (rows + pad), batch, kt.P(info))
    assert st == pykblas.KBLAS_Success
    a, b, inf = kt.to_host(dA), kt.to_host(dB), kt.to_host(info)
    assert inf.tolist() == [c + 1 for c in cols] + [0]
    # the forward sweep of the right-hand sides, as rows of the oracle's solution
    L = np.tril(po.potrf(A.T.astype(np.float64))[0])
    Bn = B.T.astype(np.float64) if side == "L" else B.astype(np.float64)   # n x nrhs
    Y = np.linalg.solve(L, Bn)
    eps = kt.EPS64 if p == "D" else kt.EPS32
    for i, c in enumerate(cols):
        k0, k1 = c // 32 * 32, min(c // 32 * 32 + 32, n)
        assert np.array_equal(a[i, k0:, k1:], a0[i, k0:, k1:], equal_nan=True), c   # [column, row]
        assert np.array_equal(a[i, :, n:], a0[i, :, n:], equal_nan=True)
        assert np.array_equal(a[i, :k0, :n], a[-1, :k0, :n])
        bi, bo = (b[i].T, b0[i].T) if side == "L" else (b[i], b0[i])
        bn, on = (bi[:n], bo[:n]) if side == "L" else (bi[:, :nrhs], bo[:, :nrhs])
        assert np.array_equal(bn[k0:], on[k0:]), c
        assert np.all(np.isnan(b[i][:, rows:]))
        if k0:
            assert np.max(np.abs(bn[:k0] - Y[:k0])) <= 64 * n * eps * max(np.max(np.abs(Y)), 1), c


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("n,nrhs", [(65, 2), (97, 1), (130, 17)])   # two, two and four waves per matrix
def test_failures_in_large_batches(h, p, n, nrhs):
    torch = kt.torch_dev()
    dt = np.float64 if p == "D" else np.float32
    few, many = 7, 2400
    A = po.gen_spd_shift_batch(62, n, few).astype(dt)
    B = po.gen_rhs_batch(72, nrhs, n, few).astype(dt)
    for i, c in ((1, 2), (3, 40), (6, n - 1)):
        A[i][c, c] = -1.0
    idx = torch.arange(many, device="cuda") % few
    out = []
    for batch, ix in ((few, torch.arange(few, device="cuda")), (many, idx)):
        dA, dB = kt.to_dev(A)[ix], kt.to_dev(B)[ix]
        info = torch.full((batch,), -7, dtype=torch.int32, device="cuda")
        st = getattr(h.lib, POSV % p)(h.h, b"R", b"L", nrhs, n, kt.P(dA), n, n * n, kt.P(dB), nrhs, nrhs * n, batch,
                                      kt.P(info))
        assert st == pykblas.KBLAS_Success
        out.append((dA, dB, info))
    (aw, bw, iw), (ag, bg, ig) = out
    assert iw.tolist() == [0, 3, 0, 41, 0, 0, n]
    assert torch.equal(iw[idx], ig) and torch.equal(bw[idx], bg)
    ok = torch.tensor([0, 2, 4, 5], device="cuda")
    ok = torch.isin(idx, ok)
    assert torch.equal(aw[idx][ok], ag[ok])
