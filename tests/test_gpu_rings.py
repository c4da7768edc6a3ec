"""The ring terms in their factored forms against the oracle's term-by-term
residuals, on amplitudes without the symmetry T_abij = T_baji and at odd sizes
(the forms use no symmetry of T2)."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SIZES = [(1, 3, 5), (3, 8, 20), (5, 17, 31)]


def plain_amplitudes(Nv, No, seed):
    rng = np.random.default_rng(seed)
    return 0.1 * rng.standard_normal((Nv, No)), 0.1 * rng.standard_normal((Nv, Nv, No, No))


def close(x, ref):
    # FP64 sums of at most a few thousand terms
    assert float(np.abs(x - ref).max()) <= 1e-11 * max(float(np.abs(ref).max()), 1e-3)


@pytest.mark.parametrize("dist", [False, True])
@pytest.mark.parametrize("size", SIZES)
def test_ccsd_rings_without_symmetry(size, dist):
    from oracle import ccsd, philox
    from sisi4s_amd import engine
    No, Nv, NG = size
    g, ei, ea = philox.system(11, No, Nv, NG)
    ints = ccsd.integrals_from_vertex(g, No)
    T1, T2 = plain_amplitudes(Nv, No, 3)
    U1, U2 = plain_amplitudes(Nv, No, 4)
    with engine.Engine(No, Nv, NG) as e:
        e.set_system(g, ei, ea)
        e.set_residual_variant(ppl=False, distinguishable=dist)
        announce("rings No=%d Nv=%d dist=%d" % (No, Nv, dist))
        R1, R2 = e.residual(1, T1, T2, slice_size=4)
        O1, O2 = ccsd.residual(1, T1, T2, g, ints, 4, ppl=False, distinguishable=dist)
        close(R1, O1)
        close(R2, O2)
        # the refinement residual in FP64 is the residual
        e.residual_anchor(T1, T2, slice_size=4)
        e.set_precision("fp64")
        R1, R2 = e.residual_refine(U1, U2, slice_size=4)
        O1, O2 = ccsd.residual(1, U1, U2, g, ints, 4, ppl=False, distinguishable=dist)
        close(R1, O1)
        close(R2, O2)


@pytest.mark.parametrize("adjacent", [False, True])
@pytest.mark.parametrize("uploaded", [False, True])
@pytest.mark.parametrize("size", SIZES)
def test_drccd_rings_without_symmetry(size, uploaded, adjacent):
    """The two-product form (vertex) and the general one (uploaded PPHH, here
    without the symmetry V_abij = V_baji) against the oracle."""
    from oracle import drccd, philox
    from sisi4s_amd import engine
    No, Nv, NG = size
    g, ei, ea = philox.system(12, No, Nv, NG)
    _, T2 = plain_amplitudes(Nv, No, 5)
    V = np.einsum("Gai,Gbj->abij", g[:, No:, :No], g[:, No:, :No])
    if uploaded:
        V = V + 0.1 * np.random.default_rng(6).standard_normal(V.shape)
    with engine.Engine(No, Nv, NG) as e:
        if uploaded:
            e.set_eigenenergies(ei, ea)
            e.set_integrals(engine.PPHH, V)
        else:
            e.set_system(g, ei, ea)
        e.set_drccd(adjacent_pairs_exchange=adjacent)
        announce("direct rings No=%d Nv=%d uploaded=%d adjacent=%d" % (No, Nv, uploaded, adjacent))
        _, R2 = e.residual(1, np.zeros((Nv, No)), T2)
    _, O2 = drccd.residual(1, T2, *drccd.integrals(V), adjacent_pairs_exchange=adjacent)
    close(R2, O2)
