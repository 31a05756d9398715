"""The step loops' near lists against whole rows: twelve steps in one loop (near lists) and in loops
of three (whole rows, dpm_api.hip: NEAR_STEPS) from one state, through in-loop rebuilds.  Both
evaluate the same interacting pairs; sums may differ in order, 1e-15 of the largest force per step,
so 1e-12 after twelve (rigid rings and FIRE likewise)."""
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


# the other loops: near lists with outputs on the last launch only (overdamped), rigid rings
@pytest.mark.parametrize("kind", ["langevin", "baoab", "brownian", "drivenBrownian", "active", "rigid_nve",
                                  "rigid_langevin", "rigid_fire"])
@pytest.mark.parametrize("interaction", ["vertexVertex", "vertexSmooth"])
def test_every_near_loop_equals_row_loops(kind, interaction):
    nrings = 40
    st = grid_state(nrings, 13, 19)
    rng = np.random.default_rng(4)
    size = 2 * float(np.mean(st["rad"]))
    pvel = rng.standard_normal((nrings, 2))
    out = []
    for chunk in (12, 3):
        g = gpu_from_state(st, potential="wca", interaction=interaction, dt=2e-3 * size,
                           particle="active" if kind == "active" else "passive")
        g.calc_neighbor_list(g.set_displacement_cutoff(0.3, size))
        if kind.startswith("rigid"):
            g.calc_rigid_force_energy()
            if kind == "rigid_nve":
                g.init_rigid_nve(1.0)
                run = g.rigid_nve
            elif kind == "rigid_langevin":
                g.init_rigid_langevin(1.0, 1.0)
                run = g.rigid_langevin
            else:
                g.init_rigid_fire([0.2, 0.5, 1.1, 0.99, 2e-3 * size, 2e-2 * size, 0.2], 20, 0)
                run = g.rigid_fire
            if kind != "rigid_langevin":
                g.set("pvel", 4.0 * pvel.ravel())
            names = ("pos", "pvel", "pangvel", "pforce", "ptorque", "force", "ppos")
        else:
            if kind == "active":
                g.set_self_propulsion(1.0, 1.0)
            elif kind != "langevin":
                g.set_noise_type(kind)
            g.calc_force_energy()
            # overdamped: F / gamma dt within a hundredth of a vertex diameter per step
            g.init_langevin(1e-2 if "rownian" in kind else 1.0, 1e3 if "rownian" in kind else 1.0, read_state=True)
            g.set("vel", np.repeat(4.0 * pvel, st["nvp"], axis=0).ravel())
            run = g.langevin
            names = ("pos", "vel", "force", "energy", "penergy", "area", "perimeter", "theta", "length", "ppos")
        for _ in range(12 // chunk):
            run(chunk)
        out.append([g.get(n) for n in names] + [g.update_count()])
        g.close()
    for n, a, b in zip(names, *out):
        assert np.all(np.isfinite(a)) and rel_err(a, b) < 1e-12, n
    assert np.array_equal(out[0][-1], out[1][-1])
