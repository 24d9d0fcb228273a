"""GPU tests of the non-uniform mixed POSV above order 64 on ill-conditioned
systems (Gaussian kernel matrices, conditions 2e5 to 6e6, some graded by four
decades on both sides): the FP32 factor and sweeps have to be as good as
substitutions for the refinement to keep its pace.

Bars: info = 0; ITER >= 0 and within 2 of the oracle's dsposv; backward error
<= 1e-13; A left as it was."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po
from test_gpu_illcond import kernel_matrix

pytestmark = pytest.mark.gpu

NS = [65, 80, 97, 112, 128, 144, 200, 256]


@pytest.mark.parametrize("side", ["L", "R"])
@pytest.mark.parametrize("nrhs", [1, 20, 64])
def test_mixed_kernel_matrices(side, nrhs):
    torch = kt.torch_dev()
    h = kt.handle()
    As = [np.asfortranarray(kernel_matrix(10 * n, n, length, shift * n, grade)) for n in NS for shift in (1e-6, 1e-7)
          for length, grade in ((0.1, 0), (0.3, 0), (0.3, -4), (0.3, 4))]
    Bs = [po.gen_rhs(172, i, *((len(A), nrhs) if side == "L" else (nrhs, len(A)))) for i, A in enumerate(As)]
    batch = len(As)
    dA, dB = [kt.to_dev(A) for A in As], [kt.to_dev(B.T) for B in Bs]
    dX = [torch.full_like(b, float("nan")) for b in dB]
    ptr = lambda ts: torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device="cuda")  # noqa: E731
    pA, pB, pX = ptr(dA), ptr(dB), ptr(dX)
    dn, dr = kt.to_dev(np.array([len(A) for A in As], np.int32)), kt.to_dev(np.full(batch, nrhs, np.int32))
    m, n = (dn, dr) if side == "L" else (dr, dn)
    mx = (max(NS), nrhs) if side == "L" else (nrhs, max(NS))
    info, it = kt.to_dev(np.full(batch, -7, np.int32)), kt.to_dev(np.full(batch, -99, np.int32))
    h.lib.kblas_sposv_vbatch_wsquery(h.h, nrhs, max(NS), batch)
    assert h.lib.kblasAllocateWorkspace(h.h) == pykblas.KBLAS_Success
    st = h.lib.kblasDsposv_vbatch(h.h, side.encode(), b"L", kt.P(m), kt.P(n), mx[0], mx[1], kt.P(pA), kt.P(dn),
                                  kt.P(pB), kt.P(m), kt.P(pX), kt.P(m), batch, kt.P(info), kt.P(it))
    assert st == pykblas.KBLAS_Success
    inf, itr = kt.to_host(info), kt.to_host(it)
    h.close()
    assert not inf.any(), inf
    want = np.array([po.sposv(side, A, B)[2] for A, B in zip(As, Bs)])
    assert np.all(itr >= 0) and np.all(np.abs(itr - want) <= 2), (itr, want)
    for i, A in enumerate(As):
        assert np.array_equal(kt.to_host(dA[i]), A), i
        assert po.solve_berr(side, A, kt.to_host(dX[i]).T, Bs[i]) <= 1e-13, i
