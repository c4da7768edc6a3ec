"""What a run is begun with, and what is changed between its iterations."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

SIZE = (3, 14, 40)


def system(seed=41):
    from oracle import ccsd, philox
    g, ei, ea = philox.system(seed, *SIZE)
    return g, ei, ea, ccsd.integrals_from_vertex(g, SIZE[0])


def linear(**kw):
    """Iterations that replace T by the estimate from its residual."""
    from sisi4s_amd import engine
    return engine.default_opts(mixer="LinearMixer", mixing_ratio=1.0, max_iterations=10,
                               level_shift=1.5, energy_convergence=0.0,
                               amplitudes_convergence=1e-12, slice_size=5, **kw)


def test_bulk_refinement_from_given_singles():
    """Singles given without doubles: the first anchor is at those singles,
    not at T = 0.  FP32 anchor: the bulk tolerance of that precision."""
    from oracle import ccsd
    from sisi4s_amd import engine
    g, ei, ea, ints = system()
    No, Nv, _ = SIZE
    T1 = 0.3 * np.random.default_rng(5).standard_normal((Nv, No))
    T2 = np.zeros((Nv, Nv, No, No))
    announce("bulk refinement from given singles")
    with engine.Engine(*SIZE) as e:
        e.set_system(g, ei, ea)
        e.ccsd_begin(linear(precision="fp32", bulk_refine_interval=8, refine_precision="fp32"),
                     T1, None)
        e.ccsd_iterate(1)
        U1, U2 = e.amplitudes()
    R1, R2 = ccsd.residual(1, T1, T2, g, ints, 5)
    O1, O2 = ccsd.estimate_amplitudes(R1, R2, T1, T2, ei, ea, 1.5)
    assert np.abs(U1 - O1).max() <= 2e-5 * np.abs(O1).max()
    assert np.abs(U2 - O2).max() <= 2e-5 * np.abs(O2).max()


def test_integrals_replaced_between_iterations():
    """From the upload of a class without the symmetry V_abij = V_baji on, the
    doubles are not projected on T_abij = T_baji."""
    from oracle import ccsd
    from sisi4s_amd import engine
    g, ei, ea, ints = system()
    No, Nv, _ = SIZE
    announce("integrals replaced between iterations")
    with engine.Engine(*SIZE) as e:
        e.set_system(g, ei, ea)
        V = e.get_integrals(engine.PPHH)
        e.ccsd_begin(linear())
        e.ccsd_iterate(2)
        T1, T2 = e.amplitudes()
        assert (T2 == T2.transpose(1, 0, 3, 2)).all()
        e.set_integrals(engine.PPHH, V + 0.05 * np.random.default_rng(7).standard_normal(V.shape))
        for _ in range(2):
            R1, R2 = e.residual(3, T1, T2, slice_size=5)
            O1, O2 = ccsd.estimate_amplitudes(R1, R2, T1, T2, ei, ea, 1.5)
            e.ccsd_iterate(1)
            T1, T2 = e.amplitudes()
            # the same residual: only the order of a few sums may differ
            assert np.abs(T1 - O1).max() <= 1e-12 * np.abs(O1).max()
            assert np.abs(T2 - O2).max() <= 1e-12 * np.abs(O2).max()
            assert np.abs(T2 - T2.transpose(1, 0, 3, 2)).max() > 1e-4


def test_any_number_of_residua():
    """maxResidua above what a run can fill is no bound."""
    from oracle import ccsd
    from sisi4s_amd import engine
    g, ei, ea, _ = system()
    kw = dict(mixer="DiisMixer", max_iterations=5, level_shift=1.5, energy_convergence=0.0,
              amplitudes_convergence=1e-12)
    announce("maxResidua 4500")
    with engine.Engine(*SIZE) as e:
        e.set_system(g, ei, ea)
        e.ccsd_solve(engine.default_opts(max_residua=4500, **kw))
        E = e.energies()
    ref = ccsd.solve(g, ei, ea, max_residua=6, **kw)
    assert np.abs(E - np.array(ref["energies"])).max() <= 1e-11 * abs(ref["energy"])
