"""FP64 / FP32 products at the edges of the kernels' block tiles (32, 64 and
128 rows) and k-chunks (16): every load mapping, odd leading dimensions (8-byte
aligned pairs), split K, and values outside the operands that must not reach
the result."""

import numpy as np
import pytest

from conftest import announce
from test_zz_no_alloc import Dev, _hip

pytestmark = pytest.mark.gpu

# tiles of 32 (small outputs), of 64 and of 128 (the last two sizes), remainders
# in m, n and k around each; K = 1..3 leave only a partial chunk
SHAPES = [(1, 1, 1), (1, 37, 5), (37, 1, 19), (16, 16, 16), (17, 15, 3), (31, 33, 17),
          (33, 65, 32), (64, 63, 47), (65, 129, 33), (127, 130, 15), (50, 50, 2500),
          (1153, 1101, 49), (4097, 4031, 37)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_products_at_tile_edges(shape, prec):
    from sisi4s_amd import engine
    lib, hip = engine.load(), _hip()
    M, N, K = shape
    # inputs rounded once to the product precision: FP32 operands are rounded
    # by the kernel, exactly representable here
    u = 2.0 ** -53 if prec == 0 else 2.0 ** -24
    rng = np.random.default_rng(M * 7 + N * 3 + K)

    def operand(rows, cols):
        """rows x cols inside a leading dimension of rows + 1 (odd for even
        rows), the padding NaN."""
        full = np.full((rows + 1, cols), np.nan)
        x = rng.standard_normal((rows, cols))
        full[:rows] = x if prec == 0 else x.astype(np.float32)
        return Dev(hip, full), full[:rows], rows + 1
    for ta in (0, 1):
        for tb in (0, 1):
            da, a, lda = operand(*((K, M) if ta else (M, K)))
            db, b, ldb = operand(*((N, K) if tb else (K, N)))
            a, b = (a.T if ta else a), (b.T if tb else b)
            ref, mag = a @ b, np.abs(a) @ np.abs(b)
            # standard bound of a length-K sum in the product precision, plus
            # the FP64 epilogue (alpha, beta) and the reference's own
            bound = (K + 2) * u * mag + (K + 4) * 2.0 ** -53 * (mag + 2.0)
            for ks in (0, 3) if K >= 48 else (0,):
                announce("gemm tile edges M=%d N=%d K=%d ta=%d tb=%d prec=%d split=%d"
                         % (M, N, K, ta, tb, prec, ks))
                dc = Dev(hip, np.ones((M, N)))
                rc = lib.sisi_gemm_device_noalloc(prec, ta, tb, M, N, K, -1.0, da.ptr, lda, db.ptr,
                                                  ldb, 2.0, dc.ptr, M, ks, None)
                assert rc == 0, lib.sisi_last_error()
                assert hip.hipDeviceSynchronize() == 0
                c = dc.read().reshape((M, N), order="F")
                dc.close()
                assert (np.abs(c - (2.0 - ref)) <= bound).all()
            da.close()
            db.close()
