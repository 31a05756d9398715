"""Step loops whose drift moves vertices farther than the cells' margin (cutoff / 3) in one step:
the next rebuild searches all vertices of the system (the reference's all-pairs list build,
cudaKernel.cuh:1735-1763) instead of the previous positions' cells, and the trajectory still
matches the oracle, which rebuilds from scratch."""
import numpy as np
import pytest
import torch

from tests.conftest import rel_err
from tests.helpers import gpu_from_state, oracle_from_state
from tests.test_oracle_rigid import ring_block

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("inter", ["vertexVertex", "vertexSmooth"])
def test_fast_rings_nve(oracle_mod, inter):
    print(f"case far_moves nve {inter}", flush=True)
    st = ring_block(gap=1.9, seed=3)
    dt = 2e-3
    o = oracle_from_state(oracle_mod, st, potential="wca", interaction=inter, costs=(1, 1, 0.1, 1), dt=dt)
    g = gpu_from_state(st, potential="wca", interaction=inter, costs=(1, 1, 0.1, 1), dt=dt)
    size = 2 * st["rad"].mean()
    cut_o = o.set_displacement_cutoff(0.5, size)
    cut_g = g.set_displacement_cutoff(0.5, size)
    o.calc_neighbor_list(cut_o)
    g.calc_neighbor_list(cut_g)
    o.calc_force_energy()
    g.calc_force_energy()
    o.init_nve(0.0)
    g.init_nve(0.0)
    # every ring translates at a speed that covers 0.6 * cutoff per step (cutoff = 0.5 size)
    rng = np.random.default_rng(1)
    speed = 0.6 * 0.5 * size / dt
    ang = rng.uniform(0, 2 * np.pi, len(st["nvp"]))
    v = np.repeat(np.c_[np.cos(ang), np.sin(ang)] * speed, st["nvp"], axis=0).ravel()
    o.set("vel", v)
    g.set("vel", v)
    for chunk in (1, 2):  # three steps: the rings meet hard soon after
        o.nve(chunk)
        g.nve(chunk)
        assert rel_err(g.get("pos"), o.get("pos"), scale=1.0) < 1e-11, chunk
        assert rel_err(g.get("force"), o.get("force")) < 1e-9, chunk
    assert g.update_count()[0] >= 2  # the list was rebuilt (all pairs) in these steps
    g.close()


@pytest.mark.parametrize("inter", ["vertexVertex", "vertexSmooth"])
def test_loop_start_far_from_list_positions(oracle_mod, inter):
    """Positions moved between loops, without a list rebuild, to 0.8 cutoff from the list positions
    (those of the last rebuild; here a translation of the whole packing, which keeps every pair
    distance): the step loop bins the list positions, whose cells allow for vertices at most
    2 cutoff / 3 away, so its start marks the system and the first rebuild searches all pairs;
    the trajectory matches the oracle, which rebuilds from scratch."""
    print(f"case far_moves loop start {inter}", flush=True)
    st = ring_block(gap=1.9, seed=5)
    dt = 2e-3
    o = oracle_from_state(oracle_mod, st, potential="wca", interaction=inter, costs=(1, 1, 0.1, 1), dt=dt)
    g = gpu_from_state(st, potential="wca", interaction=inter, costs=(1, 1, 0.1, 1), dt=dt)
    size = 2 * st["rad"].mean()
    for obj in (o, g):
        obj.calc_neighbor_list(obj.set_displacement_cutoff(0.5, size))
        obj.calc_force_energy()
        obj.init_nve(0.0)
    rng = np.random.default_rng(2)
    # rings drifting at 0.02 cutoff per step, the whole packing moved by 0.8 cutoff
    ang = rng.uniform(0, 2 * np.pi, len(st["nvp"]))
    v = np.repeat(np.c_[np.cos(ang), np.sin(ang)] * 0.02 * 0.5 * size / dt, st["nvp"], axis=0).ravel()
    shift = np.tile(0.8 * 0.5 * size * np.array([np.cos(0.7), np.sin(0.7)]), len(st["rad"]))
    for obj in (o, g):
        obj.set("pos", st["pos"] + shift)
        obj.set("vel", v)
        obj.calc_force_energy()
    u0 = g.update_count()[0]
    for chunk in (1, 4):
        o.nve(chunk)
        g.nve(chunk)
        assert rel_err(g.get("pos"), o.get("pos"), scale=1.0) < 1e-11, chunk
        assert rel_err(g.get("force"), o.get("force")) < 1e-9, chunk
    assert g.update_count()[0] > u0  # the first step rebuilt the rows (all pairs)
    g.close()


def test_fast_rigid_rings_langevin(oracle_mod):
    """Rigid Langevin (whose kick adds unit draws whatever the time step) with ring velocities that
    cover 0.6 cutoff per step: each drift flags the system as a far move, so the next rebuild
    searches all pairs; the trajectory matches the oracle, which rebuilds from scratch.  The rings
    start apart (rigid rings cannot give way: a start in contact at these speeds overlaps deeply
    within two steps and the forces blow up) and first touch in the third step, through pairs the
    far-move rebuilds found."""
    print("case far_moves rigid langevin", flush=True)
    st = ring_block(gap=4.0, seed=7)
    dt = 2e-3
    o = oracle_from_state(oracle_mod, st, potential="wca", interaction="vertexVertex", costs=(0, 0, 0, 1), dt=dt)
    g = gpu_from_state(st, potential="wca", interaction="vertexVertex", costs=(0, 0, 0, 1), dt=dt)
    size = 2 * st["rad"].mean()
    for obj in (o, g):
        obj.calc_neighbor_list(obj.set_displacement_cutoff(0.5, size))
        obj.calc_rigid_force_energy()
        obj.init_rigid_langevin(1e-2, 1.0)
    rng = np.random.default_rng(2)
    speed = 0.6 * 0.5 * size / dt
    ang = rng.uniform(0, 2 * np.pi, len(st["nvp"]))
    pv = (np.c_[np.cos(ang), np.sin(ang)] * speed).ravel()
    o.set("pvel", pv)
    g.set("pvel", pv)
    for chunk in (1, 2):
        o.rigid_loop(chunk)
        g.rigid_langevin(chunk)
        assert rel_err(g.get("pos"), o.get("pos"), scale=1.0) < 1e-11, chunk
        assert rel_err(g.get("pvel"), o.get("pvel")) < 1e-10, chunk
    assert g.update_count()[0] >= 2  # the list was rebuilt (all pairs) in these steps
    g.close()


def drifting(g, st, force, size, cutoff, dt):
    """`g` moved by 0.6 cutoff from its list positions without a list build (a translation of the whole
    packing, which keeps every pair distance), drifting on at 0.25 cutoff per `dt`; a little of the force
    in the velocities keeps FIRE's power positive.  Returns the velocities."""
    u = np.array([np.cos(0.7), np.sin(0.7)]) * cutoff * size
    g.set("pos", st["pos"] + np.tile(0.6 * u, len(st["rad"])))
    return np.tile(0.25 * u / dt, len(force) // 2) + 1e-3 * force


@pytest.mark.parametrize("inter", ["vertexVertex", "vertexSmooth"])
def test_fire_minimize_starts_beyond_displacement_test(inter):
    """A start farther than cutoff / 3 from the list positions and a first drift (below cutoff / 3 itself)
    past 2 cutoff / 3, which the cells of the list positions do not cover: FIRE on every tile (the
    library's choice for one packing of 60 rings) rebuilds as the persistent kernel does."""
    from cudaring_amd import packing
    print(f"case far_moves fire tiles {inter}", flush=True)
    st = packing.lattice_system(60, 0.8, 21, n_small=16, n_large=22, perturb=0.05)
    size = 2 * float(st["rad"].mean())
    dt = 1e-2
    out = []
    for persistent in (False, True):
        g = gpu_from_state(st, interaction=inter, costs=(1, 1, 0.1, 1))
        g.calc_neighbor_list(g.set_displacement_cutoff(0.5, size))
        g.calc_force_energy()
        g.set("vel", drifting(g, st, g.get("force"), size, 0.5, dt))
        g.calc_force_energy()
        g.init_fire((0.2, 0.5, 1.1, 0.99, dt, dt, 0.02), 20, 0)
        if persistent:
            g.set_fire_kernel(True, 0)
        g.fire_minimize(0.0, 5)
        out.append((g.get("pos"), g.get("force"), list(g.update_count())))
        g.close()
    assert out[0][2] == out[1][2] and out[0][2][0] >= 1
    assert rel_err(out[0][0], out[1][0], scale=1.0) < 1e-11
    assert rel_err(out[0][1], out[1][1]) < 1e-10


def test_rigid_fire_starts_beyond_displacement_test():
    """The same start for rigid FIRE, against a set whose list is built at the start positions."""
    print("case far_moves rigid fire", flush=True)
    st = ring_block(gap=1.5, seed=9)
    size = 2 * st["rad"].mean()
    dt = 1e-2
    out = []
    for fresh in (False, True):
        g = gpu_from_state(st, costs=(0, 0, 0, 1))
        cut = g.set_displacement_cutoff(0.5, size)
        g.calc_neighbor_list(cut)
        g.calc_rigid_force_energy()
        v = drifting(g, st, g.get("pforce"), size, 0.5, dt)
        if fresh:
            g.calc_neighbor_list(cut)
        g.calc_rigid_force_energy()
        g.init_rigid_fire([0.2, 0.5, 1.1, 0.99, dt, dt, 0.2], 20, 0)
        g.set("pvel", v)
        g.rigid_fire(5)
        out.append((g.get("pos"), g.get("pforce")))
        g.close()
    assert rel_err(out[0][0], out[1][0], scale=1.0) < 1e-11
    assert rel_err(out[0][1], out[1][1]) < 1e-10


def gradient(g, st, steps, every, seed):
    """Gradients (x0, v0, ring costs, l0) of seed . (x_N, v_N) through `steps` NVE steps."""
    nv = len(st["rad"])
    c = torch.as_tensor(np.random.default_rng(seed).standard_normal(4 * nv), device="cuda")
    ax, av = c[:2 * nv].clone(), c[2 * nv:].clone()
    gx, gv = torch.empty_like(ax), torch.empty_like(ax)
    gring = torch.empty(3 * len(st["nvp"]), dtype=torch.float64, device="cuda")
    gl0 = torch.empty(nv, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    g.nve_forward(steps, every)
    g.nve_backward(*(t.data_ptr() for t in (ax, av, gx, gv, gring, gl0)))
    return [t.cpu().numpy() for t in (gx, gv, gring, gl0)]


def test_recomputed_segment_of_fast_rings():
    """The reverse pass recomputes its segments with every system flagged for a rebuild in the first step; a
    first drift of 0.8 cutoff keeps its far-move mark, and the gradient is the one of a wide skin, whose
    recomputation makes no far move."""
    from cudaring_amd import packing
    print("case far_moves reverse pass", flush=True)
    st = packing.lattice_system(25, 0.8, 23, n_small=16, n_large=22, perturb=0.05)
    size, dt = 2 * float(st["rad"].mean()), 1e-3
    rng = np.random.default_rng(8)
    nv = len(st["rad"])
    vel = np.tile(0.8 * 0.3 * size / dt * np.array([np.cos(0.7), np.sin(0.7)]), nv) + 0.1 * rng.standard_normal(2 * nv)
    out = []
    for skin in (0.3, 2.0):
        g = gpu_from_state(st, dt=dt)
        g.calc_neighbor_list(g.set_displacement_cutoff(skin, size))
        g.set("vel", vel)
        g.calc_force_energy()
        out.append(gradient(g, st, 6, 6, 8))
        g.close()
    for a, b in zip(*out):
        assert rel_err(a, b) < 1e-11


@pytest.mark.parametrize("every", [12, 5])
def test_recomputed_segment_widens_list(every):
    """Rows built for a narrow skin serve a slow forward pass under a wide one (nothing moves past its
    displacement test); the reverse pass rebuilds them, finds rows longer than the list is wide, and
    recomputes on a wider list: the gradient is the one of rows built for the wide skin."""
    from cudaring_amd import packing
    print("case reverse pass widens list", flush=True)
    st = packing.lattice_system(25, 0.8, 23, n_small=16, n_large=22, perturb=0.05)
    size = 2 * float(st["rad"].mean())
    vel = 0.1 * np.random.default_rng(8).standard_normal(2 * len(st["rad"]))
    out = []
    for first in (0.1, 3.0):
        g = gpu_from_state(st, dt=1e-3)
        g.calc_neighbor_list(g.set_displacement_cutoff(first, size))
        w0 = g.neighbors()[1]
        g.set_displacement_cutoff(3.0, size)
        g.set("vel", vel)
        g.calc_force_energy()
        out.append(gradient(g, st, 12, every, 9))
        assert first == 3.0 or g.neighbors()[1] > w0
        g.close()
    for a, b in zip(*out):
        assert rel_err(a, b) < 1e-11
