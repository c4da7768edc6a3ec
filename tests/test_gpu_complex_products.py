"""Complex products as one launch (both planes, conjugations as signs) at sizes
around the kernels' tiles: the complex residual in FP64 and FP32 against the
oracle."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("fp32", 2e-5)])
@pytest.mark.parametrize("size", [(1, 3, 5), (4, 33, 70), (7, 31, 129)])
def test_complex_residual(size, prec, tol):
    """tol: FP64 as the other residual tests; FP32 sums of up to a few
    thousand terms of 2^-24 each, through two products in a row."""
    from oracle import ccsd_complex as cz, philox
    from sisi4s_amd import engine
    No, Nv, NG = size
    g, ei, ea = philox.system(31, No, Nv, NG)
    gz, _ = cz.gauge_transform(g.astype(complex), No, 5)
    rng = np.random.default_rng(17)

    def z(*shape):
        return 0.05 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
    T1, T2 = z(Nv, No), z(Nv, Nv, No, No)
    T2 = T2 + T2.transpose(1, 0, 3, 2)
    announce("complex products %s %s" % (size, prec))
    with engine.Engine(No, Nv, NG) as e:
        e.set_system(gz, ei, ea)
        e.set_precision(prec)
        R1, R2 = e.residual(1, T1, T2, slice_size=16)
    O1, O2 = cz.residual(1, T1, T2, gz, cz.integrals_from_vertex(gz, No), slice_size=16)
    scale = float(np.abs(O2).max())
    assert float(np.abs(R2 - O2).max()) <= tol * scale
    assert float(np.abs(R1 - O1).max()) <= tol * max(float(np.abs(O1).max()), 1e-2 * scale)
