"""FP32 products: length of the FP32 sums, seen on positive terms, where the
rounding of a chain grows with its length; and the complex products whose
outputs are too large for one launch of both planes."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(777, 640, 1531), (800, 800, 800), (250, 250, 8000),
                                   (33, 40, 5000)])
def test_chains_are_short(shape):
    """A chain of n positive terms has partial sums k mu, each rounded with at
    most u k mu / sqrt(3) rms: u sqrt(n) / 3 of the result.  K / n chains added
    in FP64 average that down by sqrt(n / K); n = 139 is the longest part a
    product of few tiles may have; factor 3 of margin (one chain of K is 3.5
    to 60 times the bound's middle at these sizes)."""
    from sisi4s_amd import engine
    M, N, K = shape
    rng = np.random.default_rng(K)
    A = rng.random((M, K)).astype(np.float32).astype(float)
    B = rng.random((K, N)).astype(np.float32).astype(float)
    announce("fp32 chains %s" % (shape,))
    C = engine.gemm(A, B, precision=engine.PRECISIONS["fp32"])
    ref = A @ B
    n = min(139, K)
    bound = 3.0 * 2.0 ** -24 * np.sqrt(n) / 3.0 * np.sqrt(n / K)
    assert np.linalg.norm(C - ref) <= bound * np.linalg.norm(ref)


def test_large_complex_outputs():
    """Outputs of 2^24 elements (Nv^2 No^2) take their planes one by one in
    FP32, the others both at once; against the FP64 residual."""
    from oracle import ccsd_complex as cz, philox
    from sisi4s_amd import engine
    No, Nv, NG = 8, 512, 4
    g, ei, ea = philox.system(33, No, Nv, NG)
    gz, _ = cz.gauge_transform(g.astype(complex), No, 5)
    rng = np.random.default_rng(3)

    def z(*shape):
        return 0.01 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
    T1, T2 = z(Nv, No), z(Nv, Nv, No, No)
    announce("large complex fp32 outputs")
    with engine.Engine(No, Nv, NG) as e:
        e.set_system(gz, ei, ea)
        R = {}
        for prec in ("fp64", "fp32"):
            e.set_precision(prec)
            R[prec] = e.residual(1, T1, T2, slice_size=64)
    for x, y in zip(R["fp32"], R["fp64"]):
        # the bulk tolerance of FP32 residuals
        assert np.abs(x - y).max() <= 2e-5 * np.abs(y).max()
