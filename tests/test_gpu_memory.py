"""Runs on a device that is almost full: the kept pair integrals are memory
that any other allocation may have."""

import ctypes
import re

import numpy as np
import pytest

from conftest import announce
from test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu

MB = 1 << 20
SIZE = (6, 120, 400)  # 0.9 GB of pair integrals


class Hog:
    """Takes all device memory but `leave` bytes."""

    def __init__(self, leave):
        self.hip, self.p = _hip(), []
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert self.hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        n = free.value - leave
        while n > 16 * MB:
            q = ctypes.c_void_p()
            if self.hip.hipMalloc(ctypes.byref(q), ctypes.c_size_t(n)) == 0:
                self.p.append(q)
                return
            self.hip.hipGetLastError()
            n -= 16 * MB

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for q in self.p:
            assert self.hip.hipFree(q) == 0


@pytest.fixture(scope="module", autouse=True)
def small_device():
    """4.5 GB for this file, once: pages that are freed are wiped (33 GB/s)
    before they can be had again."""
    with Hog(4500 * MB):
        yield


def free_memory():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def options(**kw):
    from sisi4s_amd import engine
    d = dict(mixer="DiisMixer", max_residua=6, max_iterations=9, level_shift=2.0,
             energy_convergence=0.0, amplitudes_convergence=1e-12)
    d.update(kw)
    return engine.default_opts(**d)


def engine_of(size, seed):
    from sisi4s_amd import engine
    e = engine.Engine(*size)
    e.set_system(*engine.generate_system(seed, *size))
    return e


def same(x, y):
    # kept and sliced ladder: FP64 sums in another order
    assert np.abs(np.asarray(x) - y).max() <= 1e-10 * np.abs(y).max()


@pytest.mark.parametrize("graphs", [0, 1])
def test_another_engine_takes_the_pair_integrals(graphs):
    """Between two iterations, also of a captured residual that reads them."""
    other = (8, 130, 600)
    announce("pair integrals taken by another engine, graphs=%d" % graphs)
    with engine_of(SIZE, 1) as e, engine_of(other, 2) as f:
        e.ccsd_solve(options(graphs=graphs))
        f.ccsd_solve(options())
        ref, other_ref = e.energies(), f.energies()
    with engine_of(SIZE, 1) as e:
        e.ccsd_begin(options(graphs=graphs))
        e.ccsd_iterate(4)
        with Hog(96 * MB):
            with engine_of(other, 2) as f:  # 180 MB of vertex alone
                f.ccsd_solve(options())
                same(f.energies(), other_ref)
            e.ccsd_iterate(9)
        same(e.energies(), ref)


def test_triples_take_the_pair_integrals():
    """(T) between two iterations of a run, then the rest of the run."""
    announce("pair integrals taken by (T)")
    with engine_of(SIZE, 1) as e:
        e.ccsd_begin(options())
        e.ccsd_iterate(4)
        t = e.triples()
        e.ccsd_iterate(9)
        ref = e.energies()
    with engine_of(SIZE, 1) as e:
        e.ccsd_begin(options())
        e.ccsd_iterate(4)
        with Hog(96 * MB):
            same([e.triples()], np.array([t]))
            e.ccsd_iterate(9)
        same(e.energies(), ref)


def test_next_run_on_one_engine_uses_the_idle_memory():
    """A mixed run after an FP64 run has the memory of the FP64 run's pair
    integrals; the FP64 run after it has them again."""
    announce("mixed run in the idle pair integrals")
    mixed = dict(precision="bf16x3", bulk_refine_interval=8, switch_threshold=1e-5)
    with engine_of(SIZE, 1) as e:
        e.ccsd_solve(options(**mixed))
        ref_mixed = e.energies()
        e.ccsd_solve(options())
        ref = e.energies()
    with engine_of(SIZE, 1) as e:
        e.ccsd_solve(options())
        with Hog(96 * MB):
            e.ccsd_solve(options(**mixed))
            # the reduced precision's ladder may keep its planes or not
            assert np.abs(e.energies() - ref_mixed).max() <= 1e-4 * np.abs(ref_mixed).max()
            e.ccsd_solve(options())
            same(e.energies(), ref)


def test_next_run_after_triples_keeps_pair_integrals():
    """(T) caches its operands in the idle pair integrals of the run before it;
    the next run has them whole again (the same products as the first)."""
    announce("run after (T) in the idle pair integrals")

    def flops(e):
        e.enable_stats(True)
        e.reset_stats()
        e.ccsd_solve(options())
        return e.stats()["gemm_flops"][0], e.energies()
    with engine_of(SIZE, 1) as e:
        first, ref = flops(e)
        with Hog(600 * MB):
            e.triples()
            second, E = flops(e)
        same(E, ref)
        # the build of the pair integrals included
        assert second == first


@pytest.mark.parametrize("slots,kept", [(6, True), (200, False)])
def test_pair_integrals_leave_what_the_run_needs(slots, kept):
    """0.9 of 2 GB, but not when 200 DIIS slots of 8 MB are still to come."""
    announce("pair integrals beside %d DIIS slots" % slots)
    with engine_of(SIZE, 1) as e:
        with Hog(2000 * MB):
            before = free_memory()
            e.ccsd_begin(options(max_residua=slots, max_iterations=300))
            e.ccsd_iterate(3)
            assert (before - free_memory() > 900 * MB) == kept


@pytest.mark.parametrize("width,kept", [(0, True), (6, True), (5, False)])
def test_slice_width_below_no_bounds_the_memory(width, kept):
    announce("pair integrals and slice width %d" % width)
    with engine_of(SIZE, 1) as e:
        before = free_memory()
        e.ccsd_begin(options(slice_size=width))
        e.ccsd_iterate(3)
        assert (before - free_memory() > 900 * MB) == kept


def test_threaded_batch_in_little_memory():
    """Three workers whose pair integrals do not fit together."""
    from sisi4s_amd import engine
    systems = [engine.generate_system(s, *SIZE) for s in (1, 2, 3)]
    announce("threaded batch in little memory")
    ref, _ = engine.ccsd_solve_batched(systems, options(), workers=1)
    with Hog(2500 * MB):
        E, _ = engine.ccsd_solve_batched(systems, options(), workers=3)
    same(E, np.asarray(ref))


def test_lockstep_batch_without_room_for_pair_integrals():
    """In the memory that a batch needs with sliced ladders (two iterations
    never keep pair integrals) a longer run, which would keep 134 MB of them,
    ends with the same energies."""
    from sisi4s_amd import engine
    systems = [engine.generate_system(s, 16, 56, 224) for s in (1, 2)]
    long, short = options(max_residua=2, max_iterations=4), options(max_residua=2, max_iterations=2)
    ref, _, _ = engine.ccsd_solve_lockstep(systems, long)
    for leave in range(200, 4000, 64):
        announce("lockstep batch in %d MB" % leave)
        with Hog(leave * MB):
            try:
                engine.ccsd_solve_lockstep(systems, short)
            except engine.EngineError as err:
                assert "allocation" in str(err)
                continue
            E, _, _ = engine.ccsd_solve_lockstep(systems, long)
        same(E, np.asarray(ref))
        return
    raise AssertionError("no room at all")


def test_refinement_gives_up_the_pair_integrals(monkeypatch, capfd):
    """FP32 iterations keep pair integrals, the refinement phase after them does
    not read them: their 0.9 GB count as cached when the first anchor looks
    for room for its planes."""
    monkeypatch.setenv("SISI_VERBOSE", "1")
    announce("refinement phase after plain FP32 iterations")
    with engine_of(SIZE, 1) as e:
        e.ccsd_begin(options(precision="fp32", switch_threshold=1e9, refine_interval=4,
                             refine_precision="fp32"))
        e.ccsd_iterate(4)
    said = re.findall(r"([0-9.]+) GB cached", capfd.readouterr().err)
    assert said and float(said[0]) > 0.9
