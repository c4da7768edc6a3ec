"""The ladder on kept pair integrals (plain iterations of a symmetric run)
against the oracle's driver, which slices the ladder: sizes around the 32 x 32
tiles of its packing kernels, one orbital, runs split over several calls, given
amplitudes with and without the symmetry T_abij = T_baji, the variants."""

import numpy as np
import pytest

from conftest import announce, random_amplitudes

pytestmark = pytest.mark.gpu


def options(**kw):
    d = dict(mixer="DiisMixer", max_residua=4, max_iterations=7, level_shift=1.5,
             energy_convergence=0.0, amplitudes_convergence=1e-9)
    d.update(kw)
    return d


def run(size, seed=21, initial=None, split=None, precision="fp64", **kw):
    from oracle import ccsd, philox
    from sisi4s_amd import engine
    No, Nv, NG = size
    g, ei, ea = philox.system(seed, No, Nv, NG)
    o = options(**kw)
    announce("kept ladder %s %s" % (size, kw))
    with engine.Engine(No, Nv, NG) as e:
        e.set_system(g, ei, ea)
        opts = engine.default_opts(slice_size=5, precision=precision, **o)
        a = initial if initial is not None else (None, None)
        if split is None:
            e.ccsd_solve(opts, *a)
        else:
            e.ccsd_begin(opts, *a)
            for n in split:
                e.ccsd_iterate(n)
        E, (T1, T2) = e.energies(), e.amplitudes()
    ref = ccsd.solve(g, ei, ea, slice_size=5, initial=initial, **o)
    return E, T1, T2, ref


def check(E, T1, T2, ref, tol):
    assert len(E) == len(ref["energies"])
    assert np.abs(E - np.array(ref["energies"])).max() <= tol * abs(ref["energy"])
    for x, y in ((T1, ref["T1"]), (T2, ref["T2"])):
        assert np.abs(x - y).max() <= tol * max(np.abs(y).max(), 1e-3)


# the DIIS weights of a few iterations carry FP64 rounding at most 1e4-fold
TOL = 1e-11


@pytest.mark.parametrize("size", [(1, 1, 4), (1, 5, 9), (2, 31, 40), (3, 32, 50), (4, 33, 70),
                                  (5, 65, 90)])
def test_solve(size):
    # one singles and one doubles amplitude: the overlaps of four DIIS vectors
    # in two dimensions are singular, whatever the residual
    check(*run(size, mixer="LinearMixer" if size[1] == 1 else "DiisMixer"), TOL)


def test_split_over_calls_and_linear_mixer():
    check(*run((3, 20, 40), split=(1, 1, 2, 1, 2)), TOL)
    check(*run((3, 20, 40), mixer="LinearMixer", mixing_ratio=0.7), TOL)


def test_more_vectors_than_one_reduction_launch():
    """Ten DIIS vectors: the overlaps and the combination take two launches of
    at most eight."""
    check(*run((3, 20, 40), max_residua=10, max_iterations=11), 1e-10)


def test_distinguishable_and_no_ladder():
    check(*run((3, 20, 40), distinguishable=True), TOL)
    check(*run((3, 20, 40), ppl=False), TOL)


@pytest.mark.parametrize("symmetric", [True, False])
def test_given_amplitudes(symmetric):
    """Amplitudes without the symmetry keep the sliced ladder, as they are."""
    T1, T2 = random_amplitudes(20, 3, seed=8, scale=0.02)
    if not symmetric:
        T2 = T2 + 0.02 * np.random.default_rng(9).standard_normal(T2.shape)
    check(*run((3, 20, 40), initial=(T1, T2)), TOL)


def test_fp32_iterations():
    """The product of the pairs in FP32: the bulk tolerance of that precision."""
    check(*run((4, 33, 70), precision="fp32"), 2e-5)
