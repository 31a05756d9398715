"""fire_minimize on every tile of the set (the default choice for few systems) against one persistent
workgroup per system: the same iterations to the last bit (both take their sums in the same order), a
system that stops early staying as it stopped."""
import time

import numpy as np
import pytest

from cudaring_amd import packing
from tests.conftest import rel_err
from tests.helpers import gpu_from_state, oracle_from_state, relaxed_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pot,inter,iters", [("harmonic", "vertexVertex", 30), ("wca", "vertexSmooth", 20)])
@pytest.mark.parametrize("sizes", [(60,), (64, 9), (70, 16, 40), (42,)])
def test_tiles_match_persistent(pot, inter, iters, sizes):
    systems = [relaxed_state(n, 0.8, 700 + n, final=(pot, inter)) for n in sizes]
    cat = packing.concat_systems(systems)
    sets = []
    for persistent in (None, True):
        g = gpu_from_state(cat, potential=pot, interaction=inter, costs=(1, 1, 0.1, 1),
                           rings_per_system=cat["rings_per_system"])
        g.calc_neighbor_list(g.set_displacement_cutoff(0.1, 2 * np.mean(cat["rad"])))
        g.calc_force_energy()
        dt = 0.01 * 2 * np.sqrt(np.mean(cat["a0"]) / np.pi)
        g.init_fire([0.2, 0.5, 1.1, 0.99, dt, 10 * dt, 0.2], 20, 0)
        if persistent:
            g.set_fire_kernel(True, 0)
        first = g.fire_minimize(0.0, iters)
        # a second call whose tolerance the last system meets at once
        tol = g.max_unbalanced_force()[-1] * 1.5 if len(sizes) > 1 else 0.0
        second = g.fire_minimize(tol, iters + 3)
        sets.append((g, first, second))
    (a, fa, sa), (b, fb, sb) = sets
    assert list(fa) == list(fb) == [iters] * len(sizes)
    assert list(sa) == list(sb) and (len(sizes) == 1 or sa[-1] == iters)
    for name in ("pos", "vel", "force", "energy", "l0", "area", "penergy"):
        assert np.array_equal(a.get(name), b.get(name)), name
    assert list(a.update_count()) == list(b.update_count())
    for x in (a, b):
        x.close()


def test_stopped_system_keeps_its_rows():
    """A system that meets its tolerance before it moves, displaced past the displacement test: neither
    path rebuilds its rows."""
    st = packing.lattice_system(60, 0.8, 21, n_small=16, n_large=22, perturb=0.05)
    size = 2 * float(st["rad"].mean())
    for persistent in (False, True):
        g = gpu_from_state(st)
        g.calc_neighbor_list(g.set_displacement_cutoff(0.5, size))
        last = g.get("lastpos")
        g.set("pos", st["pos"] + 0.25 * size)
        g.calc_force_energy()
        g.init_fire([0.2, 0.5, 1.1, 0.99, 1e-2, 1e-1, 0.2], 20, 0)
        if persistent:
            g.set_fire_kernel(True, 0)
        before = list(g.update_count())
        assert list(g.fire_minimize(1e9, 10)) == [0]
        assert list(g.update_count()) == before
        assert np.array_equal(g.get("lastpos"), last)
        g.close()


@pytest.mark.parametrize("persistent", [-1, 1, 0])
@pytest.mark.parametrize("tol,max_iter", [(1e9, 20), (0.0, 20)])
def test_fire_loop_goes_on_after_a_minimisation(oracle_mod, persistent, tol, max_iter):
    """fire(n) advances every system (dpmring.h), also one that a minimisation before it stopped, by its
    tolerance or by its number of iterations."""
    st = packing.lattice_system(60, 0.8, 21, n_small=16, n_large=22, perturb=0.05)
    g, o = gpu_from_state(st), oracle_from_state(oracle_mod, st)
    for s in (g, o):
        s.calc_neighbor_list(s.set_displacement_cutoff(0.5, 2 * float(st["rad"].mean())))
        s.calc_force_energy()
        s.init_fire([0.2, 0.5, 1.1, 0.99, 1e-2, 1e-1, 0.2], 20, 0)
    g.set_fire_kernel(persistent, 0)
    for s in (g, o):
        s.fire_minimize(tol, max_iter)
        s.fire(10)
    assert list(g.fire_state()["iters"]) == [10 + (0 if tol else max_iter)]
    assert rel_err(g.get("pos"), o.get("pos"), scale=1.0) < 1e-11
    g.close()


def test_choice_can_be_given_back():
    """set_fire_kernel(-1) gives the choice back to the library, and the tuner tries that choice too."""
    from cudaring_amd import autotune
    from cudaring_amd.dpm import DPMError
    st = packing.lattice_system(60, 0.8, 21, n_small=16, n_large=22, perturb=0.05)
    g = gpu_from_state(st)
    cut = g.set_displacement_cutoff(0.5, 2 * float(st["rad"].mean()))
    best, times = autotune.tune_fire(g, [0.2, 0.5, 1.1, 0.99, 1e-2, 1e-1, 0.2], cut, iters=20)
    assert "automatic" in times and len(times) == 6
    for kind in (1, -1, 0, -1):
        g.set_fire_kernel(kind, 0)
        g.init_fire([0.2, 0.5, 1.1, 0.99, 1e-2, 1e-1, 0.2], 20, 0)
        assert list(g.fire_minimize(0.0, 5)) == [5]
    for kind, waves in ((-2, 0), (2, 0), (-1, 17)):
        with pytest.raises(DPMError, match="bad argument"):
            g._chk(g.L.dpm_set_fire_kernel(g.h, kind, waves), "set_fire_kernel")
    g.close()


def test_call_on_relaxed_packing_ends_at_once():
    """A minimisation whose system has stopped does not run on to the end of its launches' chunk: on a
    packing of 200 rings that meets its tolerance at once, the tiles take a few launches more than the
    persistent kernel's one (512 launches took forty times as long; ten is allowed)."""
    st = packing.lattice_system(200, 0.8, 22, n_small=16, n_large=22, perturb=0.05)
    best = []
    for persistent in (False, True):
        g = gpu_from_state(st)
        g.calc_neighbor_list(g.set_displacement_cutoff(0.5, 2 * float(st["rad"].mean())))
        g.calc_force_energy()
        g.init_fire([0.2, 0.5, 1.1, 0.99, 1e-2, 1e-1, 0.2], 20, 0)
        if persistent:
            g.set_fire_kernel(True, 0)
        times = []
        for _ in range(6):
            t0 = time.perf_counter()
            assert list(g.fire_minimize(1e9, 10000)) == [0]
            times.append(time.perf_counter() - t0)
        best.append(min(times))
        g.close()
    assert best[0] < 10 * best[1], best
