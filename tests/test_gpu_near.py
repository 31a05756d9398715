"""The step loops' near lists against whole rows: twelve steps in one loop (near lists) and in loops
of three (whole rows, dpm_api.hip: NEAR_STEPS) from one state, through in-loop rebuilds.  Both
evaluate the same interacting pairs; sums may differ in order, 1e-15 of the largest force per step,
so 1e-12 after twelve."""
import numpy as np
import pytest

from cudaring_amd import packing
from tests.conftest import rel_err
from tests.helpers import gpu_from_state

pytestmark = pytest.mark.gpu


def grid_state(nrings, n_small, n_large):
    """Rings on a square grid, facing vertices of the largest ones 1.1 vertex diameters apart: in range
    of the attractive potentials, no overlaps that a stiff one would blow up."""
    rng = np.random.default_rng(3)
    nvp = packing.ring_sizes(nrings, n_small, n_large, rng=rng)
    a0, l0, th0, rad = packing.ring_shape_params(nvp)
    R = np.sqrt(2.0 * a0 / (nvp * np.sin(2.0 * np.pi / nvp)))
    step = 2 * R.max() + 2.2 * rad.max()
    m = int(np.ceil(np.sqrt(nrings)))
    k = np.arange(nrings)
    centers = np.stack([(k % m + 0.5) * step, (k // m + 0.5) * step], axis=1)
    pos = packing.place_rings(nvp, a0, centers, rng=rng, jitter=1e-3, l0=l0)
    return {"nvp": nvp, "box": np.array([m * step, m * step]), "pos": pos.ravel(), "rad": rad, "l0": l0,
            "theta0": th0, "a0": a0}


# 13/19: ragged tiles; 3: a ring's smallest size, 21 rings a tile; 64: one ring a tile; 4 rings: a box too
# narrow for cells, every entry kept; skin 3 with LJ range 2.5: more than one window of results
@pytest.mark.parametrize("nrings,n_small,n_large,skin,lj", [(40, 13, 19, 0.3, 1.5), (60, 3, 4, 0.5, 1.5),
                                                            (16, 64, 64, 0.2, 2.5), (4, 16, 22, 0.5, 1.5),
                                                            (40, 16, 22, 3.0, 2.5)])
@pytest.mark.parametrize("potential", ["harmonic", "lj", "adhesive"])
@pytest.mark.parametrize("interaction", ["vertexVertex", "vertexSmooth"])
def test_near_loop_equals_row_loops(nrings, n_small, n_large, skin, lj, potential, interaction):
    st = grid_state(nrings, n_small, n_large)
    rng = np.random.default_rng(4)
    vel = np.repeat(rng.standard_normal((nrings, 2)), st["nvp"], axis=0).ravel()
    size = 2 * float(np.mean(st["rad"]))
    out = []
    for chunk in (12, 3):
        g = gpu_from_state(st, potential=potential, interaction=interaction, lj=lj, dt=2e-3 * size)
        g.set("vel", 4.0 * vel)  # about a hundredth of a vertex diameter per step
        cut = g.set_displacement_cutoff(skin, size)
        g.calc_neighbor_list(cut)
        g.calc_force_energy()
        g.init_nve(1.0, read_state=True)
        for _ in range(12 // chunk):
            g.nve(chunk)
        out.append([g.get("pos"), g.get("vel"), g.get("force"), g.get("energy"), g.update_count()])
        g.close()
    for a, b in zip(out[0][:4], out[1][:4]):
        assert rel_err(a, b) < 1e-12
    assert np.array_equal(out[0][4], out[1][4])
