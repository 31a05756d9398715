"""Per-system sums against numpy on the fields they sum, for systems of one block of 2,048 vertices, of
exactly one, of one vertex more and of several, in one set.  Sums of n like-signed terms in another
order differ by at most n ulp: 1e-12 for 6,000."""
import numpy as np
import pytest

from cudaring_amd import DPMSet, packing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(2048,), (2049, 30, 2048), (6001, 2047, 64)])
def test_system_sums(counts):
    nvp, rings = [], []
    for n in counts:  # rings of 16 vertices, the last one with what is left (at least 3)
        r = [16] * ((n - 3) // 16)
        r.append(n - sum(r))
        nvp += r
        rings.append(len(r))
    nvp = np.array(nvp)
    rng = np.random.default_rng(8)
    a0, l0, th0, rad = packing.ring_shape_params(nvp)
    st = {"nvp": nvp, "box": np.tile([200.0, 190.0], len(counts)), "rad": rad, "l0": l0, "theta0": th0, "a0": a0}
    st["pos"] = packing.place_rings(nvp, a0, rng.random((len(nvp), 2)) * 190.0).ravel()
    g = DPMSet(nvp, rings_per_system=rings)
    g.load_state(st)
    g.set_types("harmonic", "vertexVertex")
    g.set_energy_costs(1, 1, 0.01, 1)
    g.set("vel", rng.standard_normal(2 * g.nv))
    g.calc_neighbor_list(g.set_displacement_cutoff(0.3, 2 * float(rad.mean())))
    g.calc_force_energy()
    v, f = g.get("vel").reshape(-1, 2), g.get("force").reshape(-1, 2)
    e, area = g.get("energy"), g.get("area")
    first = np.concatenate([[0], np.cumsum(nvp)])
    for s in range(len(counts)):
        sl = slice(g.vert_off[s], g.vert_off[s + 1])
        rl = slice(g.ring_off[s], g.ring_off[s + 1])
        disks = np.pi * (rad[first[rl]] ** 2 * (0.5 * nvp[rl] - 1)).sum()
        np.testing.assert_allclose(g.kinetic_energy()[s], 0.5 * (v[sl] ** 2).sum(), rtol=1e-12)
        np.testing.assert_allclose(g.potential_energy()[s], e[sl].sum(), rtol=1e-12)
        np.testing.assert_allclose(g.total_force_magnitude()[s], np.sqrt((f[sl] ** 2).sum() / (2 * counts[s])), rtol=1e-12)
        assert g.max_unbalanced_force()[s] == np.abs(f[sl]).max()
        np.testing.assert_allclose(g.phi()[s], (area[rl].sum() + disks) / (200.0 * 190.0), rtol=1e-12)
    g.close()
