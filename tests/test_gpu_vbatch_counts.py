"""GPU test of the non-uniform POSV above order 64 with right-hand-side counts
that ask for nothing: zero and negative counts (read on the device, so no host
check sees them) factor the matrix and leave B alone.

Bar: the factor bit for bit that of the same matrix with right-hand sides (whose
rows of the panels do not depend on them), info = 0, B untouched."""
import numpy as np
import pytest

import kbtest as kt
import pykblas
import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", ["D", "S"])
@pytest.mark.parametrize("side", ["L", "R"])
def test_posv_vbatch_counts(p, side):
    torch = kt.torch_dev()
    dt = np.float64 if p == "D" else np.float32
    n, counts, ldb = 150, [5, 0, -1, -15, -16, -17, -32, -1000], 160
    batch = len(counts)
    A = po.gen_spd_shift_batch(60, n, 1).astype(dt).repeat(batch, 0)
    dA = kt.to_dev(A)
    dB = torch.ones((batch, ldb, ldb), dtype=dA.dtype, device="cuda")
    pA, pB = kt.ptr_array(dA, batch, n * n), kt.ptr_array(dB, batch, ldb * ldb)
    i32 = lambda v: kt.to_dev(np.array(v, np.int32))  # noqa: E731
    dn, dr, lda, lb = i32([n] * batch), i32(counts), i32([n] * batch), i32([ldb] * batch)
    m, nn = (dn, dr) if side == "L" else (dr, dn)
    info = i32([-7] * batch)
    h = kt.handle()
    h.lib.kblas_posv_vbatch_wsquery(h.h, n, batch)
    assert h.lib.kblasAllocateWorkspace(h.h) == pykblas.KBLAS_Success
    st = getattr(h.lib, "kblas%sposv_vbatch" % p)(h.h, side.encode(), b"L", kt.P(m), kt.P(nn), n, n, kt.P(pA), kt.P(lda),
                                                  kt.P(pB), kt.P(lb), batch, kt.P(info))
    assert st == pykblas.KBLAS_Success
    got, inf = kt.to_host(dA), kt.to_host(info)
    h.close()
    assert not inf.any()
    assert not np.array_equal(got[0], A[0]) and bool((dB[0] != 1).any())
    for i in range(1, batch):
        assert np.array_equal(got[i], got[0]), counts[i]
        assert bool((dB[i] == 1).all()), counts[i]
