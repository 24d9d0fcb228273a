"""GPU tests of the Cholesky above order 64 on ill-conditioned SPD matrices:
Gaussian kernel matrices over sorted points, A(i,j) = exp(-(x_i - x_j)^2 / (2
l^2)), with a shift of the diagonal a few times above what the precision can
resolve (conditions about 1e13 in FP64, 1e6 in FP32), some graded on both sides
by a diagonal that spans four decades.  The 16 x 16 diagonal tiles of their
factors have conditions up to 1e6, where products with a tile's inverse lose
what substitution keeps.

Bars: info = 0 (LAPACK factors each of them); the factor's error element by
element, |L L^T - A|(i,j) <= (n / 2 + 8) eps sqrt(A(i,i) A(j,j)): the bound
(n + 1) (eps / 2) |L| |L^T| of a Cholesky factorization with substitutions, with
Cauchy-Schwarz, and a few roundings for the reciprocals; normwise backward error
of the solution <= 4 n eps."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po

pytestmark = pytest.mark.gpu

NS = [65, 80, 97, 128, 200, 256]


@pytest.fixture(scope="module")
def h():
    hh = kt.handle()
    yield hh
    hh.close()


def prec(p):
    return (np.float64, kt.EPS64) if p == "D" else (np.float32, kt.EPS32)


def kernel_matrix(seed, n, length, shift, grade):
    x = np.sort(np.random.default_rng(seed).random(n))
    A = np.exp(-(x[:, None] - x[None, :]) ** 2 / (2 * length * length)) + shift * np.eye(n)
    d = 10.0 ** np.linspace(0, grade, n)
    return A * np.outer(d, d)


def kernel_batch(n, dt):
    shift = 5e-13 if dt == np.float64 else 2.5e-8 * n
    out = [kernel_matrix(10 * n + s, n, length, shift, grade)
           for length, grade in ((0.1, 0), (0.3, 0), (0.3, -4), (0.3, 4)) for s in range(2)]
    return np.array(out).astype(dt).astype(np.float64)


def check_factor(A, got, eps, what):
    n = len(A)
    L = np.tril(got.astype(np.longdouble))
    d = np.sqrt(np.diag(A))
    err = float(np.max(np.abs(L @ L.T - A) / np.outer(d, d))) / eps
    assert err <= n / 2 + 8, (what, err)


def run(h, p, side, A, nrhs, reps):
    """POTRF (nrhs = 0) or POSV of the symmetric matrices A, each reps times over"""
    torch = kt.torch_dev()
    dt, eps = prec(p)
    few, n = A.shape[:2]
    batch = few * reps
    dA = kt.to_dev(A.astype(dt)).repeat(reps, 1, 1)
    info = torch.full((batch,), -7, dtype=torch.int32, device="cuda")
    dB = B = None
    if nrhs:
        rows, cols = (n, nrhs) if side == "L" else (nrhs, n)
        B = po.gen_rhs_batch(170 + nrhs, rows, cols, few).astype(dt).astype(np.float64)
        dB = kt.to_dev(B.astype(dt)).repeat(reps, 1, 1)
        st = getattr(h.lib, "kblas%sposv_batch_strided" % p)(h.h, side.encode(), b"L", rows, cols, kt.P(dA), n, n * n,
                                                             kt.P(dB), rows, rows * cols, batch, kt.P(info))
    else:
        st = getattr(h.lib, "kblas%spotrf_batch_strided" % p)(h.h, b"L", n, kt.P(dA), n, n * n, batch, kt.P(info))
    assert st == pykblas.KBLAS_Success
    assert int((info != 0).sum()) == 0, info.unique()
    Lh = kt.to_host(dA[batch - few:])
    for i in range(few):
        check_factor(A[i], Lh[i].T, eps, i)
    if nrhs:
        Xh = kt.to_host(dB[batch - few:])
        for i in range(few):
            assert po.solve_berr(side, A[i], Xh[i].T, B[i].T) <= 4 * n * eps, i


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("n", NS)
@pytest.mark.parametrize("side,nrhs", [("R", 0), ("L", 1), ("R", 5), ("R", 33), ("L", 63)])
def test_four_waves(h, p, n, side, nrhs):
    dt, _ = prec(p)
    run(h, p, side, kernel_batch(n, dt), nrhs, 1)


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("n,side,nrhs", [(65, "R", 0), (97, "R", 17), (128, "L", 30), (200, "R", 0), (200, "R", 4)])
def test_two_waves(h, p, n, side, nrhs):
    """batches of more than 1,024 matrices run two waves per matrix"""
    dt, _ = prec(p)
    run(h, p, side, kernel_batch(n, dt), nrhs, 129)


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("nrhs", [3, 40])
def test_nonuniform(h, p, nrhs):
    torch = kt.torch_dev()
    dt, eps = prec(p)
    As = [A for n in NS for A in kernel_batch(n, dt)]
    Bs = [po.gen_rhs(171, i, nrhs, len(A)).astype(dt).astype(np.float64) for i, A in enumerate(As)]
    dA = [kt.to_dev(A.astype(dt)) for A in As]
    dB = [kt.to_dev(B.T.astype(dt)) for B in Bs]
    batch = len(As)
    ptr = lambda ts: torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device="cuda")  # noqa: E731
    pA, pB = ptr(dA), ptr(dB)
    dn, dr = kt.to_dev(np.array([len(A) for A in As], np.int32)), kt.to_dev(np.full(batch, nrhs, np.int32))
    info = kt.to_dev(np.full(batch, -7, np.int32))
    h.lib.kblas_posv_vbatch_wsquery(h.h, max(NS), batch)
    assert h.lib.kblasAllocateWorkspace(h.h) == pykblas.KBLAS_Success
    st = getattr(h.lib, "kblas%sposv_vbatch" % p)(h.h, b"R", b"L", kt.P(dr), kt.P(dn), nrhs, max(NS), kt.P(pA), kt.P(dn),
                                                  kt.P(pB), kt.P(dr), batch, kt.P(info))
    assert st == pykblas.KBLAS_Success
    inf = kt.to_host(info)
    assert not inf.any(), inf
    for i, A in enumerate(As):
        check_factor(A, kt.to_host(dA[i]).T, eps, i)
        assert po.solve_berr("R", A, kt.to_host(dB[i]).T, Bs[i]) <= 4 * len(A) * eps, i
