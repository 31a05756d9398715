"""Rings that reach past half the box from their centre: the reference takes every vertex's position
relative to the ring's centre as a minimum image (getRelativeVertexPos, cudaKernel.cuh:273-279), so their
segments jump by a box length there.  The step loops give the forces that the single force call gives, and
the oracle's trajectory; also for rings just inside (elongated, longer than a quarter of the box)."""
import numpy as np
import pytest

from cudaring_amd import packing
from tests.conftest import rel_err
from tests.helpers import gpu_from_state, oracle_from_state

pytestmark = pytest.mark.gpu


def state(n, reach):
    """A ring of n vertices of radius `reach` box lengths and a small one, side by side as they come."""
    nvp = np.array([n, 12])
    a0, l0, th0, rad = packing.ring_shape_params(nvp)
    R = np.sqrt(2.0 * a0[0] / (n * np.sin(2.0 * np.pi / n)))
    L = R / reach
    pos = packing.place_rings(nvp, a0, np.array([[0.55 * L, 0.45 * L], [0.1 * L, 0.9 * L]]),
                              rng=np.random.default_rng(3), jitter=1e-2, l0=l0)
    return {"nvp": nvp, "box": np.array([L, 1.1 * L]), "pos": pos.ravel(), "rad": rad, "l0": l0, "theta0": th0, "a0": a0}


# radius in box lengths: 0.2 (past a quarter of the box from the first vertex, within one from the middle),
# 0.3 (past that, within half from the centre), 0.47 and 0.53 (about the line), 0.6; 40 vertices in one
# tile, 90 in two slices
@pytest.mark.parametrize("reach", [0.2, 0.3, 0.47, 0.53, 0.6])
@pytest.mark.parametrize("n", [40, 90])
@pytest.mark.parametrize("inter", ["vertexVertex", "vertexSmooth"])
def test_loops_give_the_force_call(oracle_mod, n, reach, inter):
    st = state(n, reach)
    size = 2 * float(st["rad"].mean())
    g, o = gpu_from_state(st, interaction=inter), oracle_from_state(oracle_mod, st, interaction=inter)
    for s in (g, o):
        s.calc_neighbor_list(s.set_displacement_cutoff(0.5, size))
        s.calc_force_energy()
        s.init_nve(0.0)
    for steps in (8, 3):  # near lists, whole rows
        g.nve(steps)
        o.nve(steps)
        assert rel_err(g.get("pos"), o.get("pos"), scale=1.0) < 1e-11
        force = g.get("force")
        assert rel_err(force, o.get("force")) < 1e-10
        g.calc_force_energy()
        assert rel_err(force, g.get("force")) < 1e-11
    g.close()
