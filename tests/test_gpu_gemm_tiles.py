"""FP64 / FP32 products at the edges of the kernels' block tiles (32, 64 and
128 rows) and k-chunks (16): every load mapping, odd leading dimensions (8-byte
aligned pairs), split K, and values outside the operands that must not reach
the result."""

import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

# tiles of 32 (small outputs), of 64 and of 128 (the last two sizes), remainders
# in m, n and k around each; K = 1..3 leave only a partial chunk
SHAPES = [(1, 1, 1), (1, 37, 5), (37, 1, 19), (16, 16, 16), (17, 15, 3), (31, 33, 17),
          (33, 65, 32), (64, 63, 47), (65, 129, 33), (127, 130, 15), (50, 50, 2500),
          (1153, 1101, 49), (4097, 4031, 37)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_products_at_tile_edges(shape, prec):
    import torch
    from sisi4s_amd import engine
    lib = engine.load()
    M, N, K = shape
    # inputs rounded once to the product precision: FP32 operands are rounded
    # by the kernel, exactly representable here
    u = 2.0 ** -53 if prec == 0 else 2.0 ** -24
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N * 3 + K)

    def operand(rows, cols):
        """Column-major rows x cols inside a leading dimension of rows + 1
        (odd for even rows), the padding NaN."""
        full = torch.full((cols, rows + 1), float("nan"), device="cuda", dtype=torch.float64)
        x = torch.randn(cols, rows, generator=g, device="cuda", dtype=torch.float64)
        full[:, :rows] = x if prec == 0 else x.float().double()
        return full, full[:, :rows].T
    for ta in (0, 1):
        for tb in (0, 1):
            fa, a = operand(K if ta else M, M if ta else K)
            fb, b = operand(N if tb else K, K if tb else N)
            a, b = (a.T if ta else a), (b.T if tb else b)
            ref, mag = a @ b, a.abs() @ b.abs()
            for ks in (0, 3) if K >= 48 else (0,):
                announce("gemm tile edges M=%d N=%d K=%d ta=%d tb=%d prec=%d split=%d"
                         % (M, N, K, ta, tb, prec, ks))
                c = torch.ones(N, M, device="cuda", dtype=torch.float64)
                rc = lib.sisi_gemm_device_noalloc(
                    prec, ta, tb, M, N, K, -1.0, fa.data_ptr(), fa.shape[1], fb.data_ptr(),
                    fb.shape[1], 2.0, c.data_ptr(), M, ks,
                    torch.cuda.current_stream().cuda_stream)
                assert rc == 0, lib.sisi_last_error()
                torch.cuda.synchronize()
                # standard bound of a length-K sum in the product precision,
                # plus the FP64 epilogue (alpha, beta) and the reference's own
                bound = (K + 2) * u * mag + (K + 4) * 2.0 ** -53 * (mag + 2.0)
                assert bool(((c.T - (2.0 - ref)).abs() <= bound).all())
