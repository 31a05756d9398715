"""Workloads of the deformable-ring engine, from one force evaluation of a small packing to the
largest active system, through the public entry points of cudaring_amd.

`listed()` names the standing cases and `draw(rng)` gives more of the same ranges.  `prepare`
makes a packing from a seed and the DPMSet that a program would hold, `run` is one pass through
the entry points, `work` counts what a pass cannot do without, and `exact` gives the outputs as
plain torch computes them in 64 bits, without the engine.
"""
import math

import numpy as np
import torch

KWCA = 1.122462048
PI = math.pi
DEV = "cuda"
F64 = torch.float64


# ------------------------------------------------------------------------------ the cases
# kind "md": a stretch of an integrator's loop and the energies a driver logs after it
# kind "rigid": the same for rigid rings; kind "fire": a compression cycle (grow, minimise,
# shrink back, minimise) of one or many packings; kind "grad": a trajectory differentiated
# through torch; kind "setup": neighbour list, forces and energies of a loaded packing.
BIDISPERSE = {"n_small": 16, "n_large": 22}
EQUAL32 = {"n_small": 32, "n_large": 32}


def listed():
    return [
        # the small NVE run of the benchmark: 608 vertices, where only latency counts
        {"name": "nve_32", "kind": "md", "systems": 1, "rings": 32, **BIDISPERSE, "pot": "harmonic",
         "inter": "vertexVertex", "noise": "nve", "steps": 100, "tune": False},
        # one step per call, as a program that looks at every step (or drives another loop) does
        {"name": "step_call_256", "kind": "md", "systems": 1, "rings": 256, **EQUAL32, "pot": "harmonic",
         "inter": "vertexSmooth", "noise": "langevin", "steps": 1, "tune": False},
        # the benchmark's thermostatted run between two lines of the energy log
        {"name": "nvt_1024", "kind": "md", "systems": 1, "rings": 1024, **BIDISPERSE, "pot": "wca",
         "inter": "vertexSmooth", "noise": "langevin", "steps": 100, "tune": True},
        # an overdamped run of 32-vertex rings, the ring size of the run drivers
        {"name": "brownian_2000", "kind": "md", "systems": 1, "rings": 2000, **EQUAL32, "pot": "wca",
         "inter": "vertexSmooth", "noise": "brownian", "steps": 50, "tune": False},
        # an ensemble of independent thermostatted packings in one set
        {"name": "ensemble_64x61", "kind": "md", "systems": 64, "rings": 61, **BIDISPERSE, "pot": "harmonic",
         "inter": "vertexVertex", "noise": "baoab", "steps": 50, "tune": False},
        # the large active adhesive monolayer, 524,288 vertices: throughput counts
        {"name": "active_16384", "kind": "md", "systems": 1, "rings": 16384, **EQUAL32, "pot": "adhesive",
         "inter": "vertexSmooth", "noise": "active", "steps": 20, "tune": True},
        # the benchmark packing as rigid rings
        {"name": "rigid_1024", "kind": "rigid", "systems": 1, "rings": 1024, **BIDISPERSE, "pot": "wca",
         "inter": "vertexSmooth", "steps": 100},
        # batched compression of many packings of 16 to 256 rings
        {"name": "fire_512", "kind": "fire", "systems": 512, "rings": 256, **BIDISPERSE, "iters": 60, "host": False},
        # one packing at a time, as compressFIRE runs
        {"name": "fire_1", "kind": "fire", "systems": 1, "rings": 200, **BIDISPERSE, "iters": 100, "host": False},
        # the driver's loop with a host check after every iteration, on makeDPM's 32 rings of 32
        {"name": "fire_check_32", "kind": "fire", "systems": 1, "rings": 32, **EQUAL32, "iters": 10, "host": True},
        # gradients of a trajectory with respect to state and parameters, forward and backward
        {"name": "grad_256", "kind": "grad", "systems": 1, "rings": 256, **BIDISPERSE, "pot": "harmonic",
         "inter": "vertexVertex", "steps": 100, "every": 50},
        # what every driver does after reading a packing: list, forces, energies
        {"name": "setup_1024", "kind": "setup", "systems": 1, "rings": 1024, **BIDISPERSE, "pot": "wca",
         "inter": "vertexSmooth"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["md", "md", "md", "rigid", "fire", "fire", "grad", "setup"])
    size = dict(rng.choice([BIDISPERSE, EQUAL32, {"n_small": 13, "n_large": 19}, {"n_small": 24, "n_large": 33}]))
    pot, inter = rng.choice(["harmonic", "wca", "adhesive", "lj"]), rng.choice(["vertexVertex", "vertexSmooth"])
    if kind == "md":
        noise = rng.choice(["nve", "langevin", "baoab", "brownian", "active"])
        rings = _log_int(rng, 24, 12000)
        systems = rng.choice([1, 1, rng.randint(2, 48)])
        rings = max(20, rings // systems) if systems > 1 else rings
        return {"kind": kind, "systems": systems, "rings": rings, **size, "pot": pot, "inter": inter, "noise": noise,
                "steps": rng.choice([1, 7, 20] if rings * systems > 2000 else [1, 25, 100]), "tune": False}
    if kind == "rigid":
        return {"kind": kind, "systems": 1, "rings": _log_int(rng, 24, 4000), **size, "pot": rng.choice(["harmonic", "wca"]),
                "inter": inter, "steps": rng.choice([1, 20, 100])}
    if kind == "fire":
        systems = rng.choice([1, _log_int(rng, 2, 300)])
        host = systems == 1 and rng.random() < 0.3
        return {"kind": kind, "systems": systems, "rings": rng.randint(16, 256), **size,
                "iters": 10 if host else rng.randint(20, 80), "host": host}
    if kind == "grad":
        return {"kind": kind, "systems": 1, "rings": _log_int(rng, 24, 600), **size, "pot": "harmonic", "inter": inter,
                "steps": rng.randint(20, 90), "every": rng.choice([10, 25, 50])}
    return {"kind": kind, "systems": rng.choice([1, rng.randint(2, 40)]), "rings": rng.randint(16, 1200), **size, "pot": pot,
            "inter": inter}


# --------------------------------------------------------------------------- the packing
def _sites(rows, cols):
    """The 18 sites of the first two shells around every site of a periodic triangular lattice
    (even number of rows; odd rows shifted by half a spacing): their index and their offset."""
    r, c = np.divmod(np.arange(rows * cols), cols)
    idx, off = [], []
    for dr in (-2, -1, 0, 1, 2):
        for dc in range(-3, 4):
            shift = 0.5 * ((r + dr) % 2 - r % 2)
            x, y = dc + shift, np.full(r.shape, dr * math.sqrt(0.75))
            d = x * x + y * y
            keep = (d > 0.5) & (d < 4.5)
            idx.append(np.where(keep, ((r + dr) % rows) * cols + (c + dc) % cols, -1))
            off.append(np.stack([x, y], -1))
    idx, off = np.stack(idx, 1), np.stack(off, 1)
    take = np.argsort(idx < 0, axis=1, kind="stable")[:, :18]
    return np.take_along_axis(idx, take, 1), np.take_along_axis(off, take[..., None], 1)


def _ring_counts(case):
    if case["kind"] == "fire" and case["systems"] > 1:  # packings of 16 rings up to the case's number
        lo, hi = 16, case["rings"]
        return [lo + (hi - lo) * ((7 * k) % case["systems"]) // max(1, case["systems"] - 1) for k in range(case["systems"])]
    return [case["rings"]] * case["systems"]


def packing(case, seed):
    """Confluent rings: power-diagram cells of a jittered triangular lattice (vacancies where the
    ring count does not fill it), pulled back by half the gap to each neighbour, corners rounded,
    cut into segments of equal length.  Neighbouring walls stand at about the potential's contact
    distance; rest areas and lengths are the initial ones, as in a relaxed packing.  Flat tensors
    on the GPU."""
    rng = np.random.default_rng(seed)
    gap = {"wca": 1.10, "lj": 1.12, "harmonic": 0.985, "adhesive": 1.0}[case.get("pot", "harmonic")]
    counts = _ring_counts(case)
    cx, nn, nb, off, box, sizes = [], [], [], [], [], []
    base = 0
    for N in counts:
        rows = max(4, 2 * int(round(math.sqrt(N * 2 / math.sqrt(3)) / 2)))
        cols = max(4, -(-N // rows))
        ring_of = np.full(rows * cols + 1, -1)
        ring_of[np.sort(rng.permutation(rows * cols)[:N])] = np.arange(N)
        site = np.flatnonzero(ring_of[:-1] >= 0)
        idx, o = _sites(rows, cols)
        n = np.where(rng.permutation(N) < N // 2, case["n_large"], case["n_small"])
        a = 1.30
        jit = 0.06 * a * (2 * rng.random((rows * cols, 2)) - 1)
        r, c = np.divmod(site, cols)
        cx.append(np.stack([(c + 0.5 * (r % 2) + 0.25) * a, (r + 0.5) * a * math.sqrt(0.75)], -1) + jit[site])
        nbr = np.where(idx[site] >= 0, ring_of[idx[site]], -1)
        d = o[site] * a + np.where((idx[site] >= 0)[..., None], jit[idx[site]], 0) - jit[site][:, None]
        nb.append(np.where(nbr >= 0, nbr + base, -1))
        off.append(d)
        big = n == case["n_large"] if case["n_small"] != case["n_large"] else rng.permutation(N) < N // 2
        ratio = case["n_large"] / case["n_small"] if case["n_small"] != case["n_large"] else 1.4
        sizes.append(0.5 * a * np.where(big, ratio, 1.0) * 2 / (1 + ratio))
        nn.append(n)
        box.append([cols * a, rows * a * math.sqrt(0.75)])
        base += N
    t = lambda v, k=F64: torch.as_tensor(np.concatenate(v), dtype=k, device=DEV)  # noqa: E731
    cen, nbr, off, R = t(cx), t(nb, torch.int64), t(off), t(sizes)
    nvp_np = np.concatenate(nn).astype(np.int64)
    nvp = torch.as_tensor(nvp_np, device=DEV)
    NR, fine = len(nvp_np), 256
    has = nbr >= 0
    D = off.norm(dim=-1)
    ang = torch.atan2(off[..., 1], off[..., 0])
    bis = 0.5 * D + (R[:, None] ** 2 - torch.where(has, R[nbr.clamp(min=0)], R[:, None]) ** 2) / (2 * D)
    th = torch.arange(fine, device=DEV, dtype=F64) * (2 * PI / fine)
    rad = PI * R * 0.92 / nvp
    most = int(nvp_np.max())
    k = torch.arange(most, device=DEV)
    phase = torch.as_tensor(rng.random(NR), device=DEV)
    xy = None
    for _ in range(2):
        room = bis - 0.5 * gap * (rad[:, None] + rad[nbr.clamp(min=0)])
        room = torch.where(has, room, torch.full_like(room, 9.0))
        cap = 1.2 * room.min(dim=1).values
        rr = cap[:, None].expand(NR, fine).clone()
        for q in range(room.shape[1]):
            cs = torch.cos(th[None] - ang[:, q, None])
            rr = torch.minimum(rr, torch.where(cs > 0.1, room[:, q, None] / cs.clamp(min=0.1), rr))
        px, py = rr * torch.cos(th), rr * torch.sin(th)
        sx, sy = px.roll(-1, 1) - px, py.roll(-1, 1) - py
        arc = torch.cumsum(torch.sqrt(sx * sx + sy * sy), 1)
        total = arc[:, -1]
        at = ((k[None] + phase[:, None]) % nvp[:, None]) * (total / nvp)[:, None]
        j = torch.searchsorted(arc, at.contiguous()).clamp(max=fine - 1)
        before = torch.where(j > 0, arc.gather(1, (j - 1).clamp(min=0)), torch.zeros_like(at))
        f = (at - before) / (arc.gather(1, j) - before)
        xy = torch.stack([px.gather(1, j) + f * sx.gather(1, j), py.gather(1, j) + f * sy.gather(1, j)], -1)
        ok = k[None] < nvp[:, None]
        nxt = torch.where(k[None] + 1 < nvp[:, None], k[None] + 1, torch.zeros_like(k)[None])
        seg = (xy.gather(1, nxt[..., None].expand_as(xy)) - xy).norm(dim=-1) * ok
        l0r = seg.sum(1) / nvp
        rad = 0.5 * l0r
    # vertices of a ring in counter-clockwise order from its first one
    first_angle = torch.argsort(torch.where(ok, (k[None] + phase[:, None]) % nvp[:, None], torch.full_like(seg, 1e9)), 1)
    xy = xy.gather(1, first_angle[..., None].expand_as(xy))
    pos = (xy + cen[:, None])[ok]
    ring = torch.arange(NR, device=DEV)[:, None].expand(NR, most)[ok]
    noise = torch.as_tensor(rng.standard_normal((int(nvp_np.sum()), 2)), device=DEV)
    pos = pos + 4e-3 * l0r[ring][:, None] * noise
    first = torch.cumsum(nvp, 0) - nvp
    nv = pos.shape[0]
    v = torch.arange(nv, device=DEV)
    nx = torch.where(v + 1 == (first + nvp)[ring], first[ring], v + 1)
    pv = torch.where(v == first[ring], (first + nvp - 1)[ring], v - 1)
    rel = pos - cen[ring]
    shoe = rel[:, 0] * rel[nx, 1] - rel[nx, 0] * rel[:, 1]
    area = 0.5 * torch.zeros(NR, dtype=F64, device=DEV).index_put_((ring,), shoe, accumulate=True)
    # rounded to single precision: the sum above may round its last bit either way
    a0 = area.float().double()
    T = {"nve": 1e-3, "active": 1e-4}.get(case.get("noise"), 1e-3 if case["kind"] == "grad" else 1e-2)
    vel = (torch.as_tensor(rng.standard_normal((NR, 2)), device=DEV) * math.sqrt(T))[ring]
    sysr = np.repeat(np.arange(len(counts)), counts)
    return {"pos": pos, "vel": vel, "rad": rad[ring], "l0": l0r[ring], "theta0": (2 * PI / nvp.double())[ring], "a0": a0,
            "box": np.array(box), "nvp": nvp_np, "counts": counts, "ring": ring, "next": nx, "prev": pv, "first": first,
            "sys_of_ring": torch.as_tensor(sysr, device=DEV), "ring_nb": nbr, "T": T,
            "angle": torch.as_tensor(rng.uniform(-PI, PI, NR), device=DEV),
            "unit": float(2 * np.sqrt(float(a0.mean()) / PI)), "size": 2 * float(rad[ring].float().mean()),
            "grad_x": torch.as_tensor(rng.standard_normal(2 * nv), device=DEV) if case["kind"] == "grad" else None}


GAMMA = 1.0
FIRE = (0.1, 0.5, 1.1, 0.99, 0.01, 0.1, 0.1)  # a_start, f_dec, f_inc, f_a, dt, dt_max, a
DPHI, TOL = 1e-3, 1e-12


def _settings(case, p):
    """Shape costs, skin, time step and driving of the case's run."""
    kind, noise = case["kind"], case.get("noise")
    if noise == "active":  # the active driver's costs and units
        q = {"costs": (1e5, 20.0, 10.0, 1.0), "skin": 0.5, "dt": 1e-3 * p["unit"], "gamma": GAMMA / p["unit"],
             "driving": 0.1 * GAMMA / p["unit"], "taup": 100.0 * p["unit"]}
    elif kind == "fire":
        q = {"costs": (1.0, 1.0, 0.1, 1.0), "skin": 0.3, "dt": 0.01, "gamma": GAMMA}
    elif noise == "nve" or kind == "grad":
        soft = case["pot"] == "harmonic"
        q = {"costs": (1.0, 1.0, 0.01, 1.0), "skin": 0.3, "dt": (0.01 if soft else 1e-3) * p["unit"], "gamma": GAMMA}
    else:
        q = {"costs": (1.0, 1.0, 0.01, 1.0), "skin": 0.5, "dt": 1e-3 * p["unit"], "gamma": GAMMA}
    if noise == "brownian":
        q["dt"] = 1e-5 * p["unit"]
    return q


def prepare(case, seed):
    from cudaring_amd import DPMSet, autotune
    p = packing(case, seed)
    q = _settings(case, p)
    s = DPMSet(p["nvp"], rings_per_system=p["counts"])
    host = {k: p[k].reshape(-1).cpu().numpy() for k in ("pos", "vel", "rad", "l0", "theta0", "a0")}
    s.load_state({**host, "box": p["box"].ravel()})
    noise = case.get("noise")
    s.set_types(case.get("pot", "harmonic"), case.get("inter", "vertexVertex"), particle="active" if noise == "active" else "passive")
    if case.get("pot") == "lj":
        s.set_lj_cutoff(1.5)
    if case.get("pot") == "adhesive":
        s.set_attraction(0.1, 0.2)
    s.set_energy_costs(*q["costs"])
    s.set_dt(q["dt"])
    s.set_seed(seed + 17)
    if noise == "active":
        s.set_self_propulsion(q["driving"], q["taup"])
    cut = s.set_displacement_cutoff(q["skin"], p["size"])
    s.calc_neighbor_list(cut)
    state = {"s": s, "case": case, "cut": cut}
    if case["kind"] == "md":
        s.calc_force_energy()
        if noise in ("baoab", "brownian"):
            s.set_noise_type(noise)
        if noise == "nve":
            s.init_nve(p["T"], read_state=True)
        else:
            s.init_langevin(p["T"], q["gamma"], read_state=True)
        if case["tune"]:
            autotune.tune_waves_per_tile(s, reps=20)
        if noise == "active":
            s.set("pangle", p["angle"].cpu().numpy())
    elif case["kind"] == "rigid":
        s.set("prad", np.sqrt(host["a0"] / PI))
        s.init_rigid_nve(p["T"], read_state=True)
        s.set("pvel", p["vel"][p["first"]].reshape(-1).cpu().numpy())
        s.calc_rigid_force_energy()
    elif case["kind"] == "fire":
        s.calc_force_energy()
    elif case["kind"] == "grad":
        from cudaring_amd.autograd import DPMAdjoint
        nr = s.np
        state["adj"] = DPMAdjoint(s, cut)
        state["in"] = [p["pos"].reshape(-1), p["vel"].reshape(-1), *(torch.full((nr,), c, dtype=F64, device=DEV)
                                                                    for c in q["costs"][:3]), p["l0"]]
        state["gx"] = p["grad_x"]
    return state


class _Buffer:
    """A device array of the set, for torch to look at; it keeps the set, which owns the memory."""

    def __init__(self, s, ptr, n):
        self.owner = s
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (ptr, False), "version": 2}


def _field(s, name):
    n = s.field_size(name)
    if name in ("pos", "vel", "force", "pvel", "ppos", "pforce"):
        return [torch.as_tensor(_Buffer(s, s.device_ptr(name, k), n // 2), device=DEV) for k in (0, 1)]
    return torch.as_tensor(_Buffer(s, s.device_ptr(name), n), device=DEV)


def run(state):
    s, case = state["s"], state["case"]
    kind = case["kind"]
    if kind == "md":
        (s.nve if case["noise"] == "nve" else s.langevin)(case["steps"])
        out = {"epot": s.potential_energy(), "ekin": s.kinetic_energy(), "pos": _field(s, "pos"), "vel": _field(s, "vel"),
               "force": _field(s, "force")}
        if case["noise"] == "active":
            out["angle"] = _field(s, "pangle")
        return out
    if kind == "rigid":
        s.rigid_nve(case["steps"])
        return {"ekin": s.rigid_kinetic_energy(), "pos": _field(s, "pos"), "pvel": _field(s, "pvel"), "omega": _field(s, "pangvel"),
                "pforce": _field(s, "pforce"), "angle": _field(s, "pangle")}
    if kind == "fire":
        force, grown = [], None
        for way in (1, -1):
            if way == 1:
                phi = s.phi()
                grown = np.sqrt((phi + DPHI) / phi)
            s.scale_vertices(grown if way == 1 else 1.0 / grown)
            s.calc_neighbor_list(state["cut"])
            s.calc_force_energy()
            s.reset_last_positions()
            s.init_fire(FIRE, 20, 0)
            if case["host"]:  # one iteration and one look at the forces per turn
                for _ in range(case["iters"]):
                    s.fire(1)
                    if s.max_unbalanced_force()[0] <= TOL:
                        break
            else:
                s.fire_minimize(TOL, case["iters"])
            force.append(s.total_force_magnitude())
        return {"force_size": force, "epot": s.potential_energy(), "pos": _field(s, "pos"), "vel": _field(s, "vel"),
                "force": _field(s, "force"), "l0": _field(s, "l0")}
    if kind == "grad":
        leaves = [x.clone().requires_grad_() for x in state["in"]]
        xN, vN = state["adj"].trajectory(*leaves, case["steps"], case["every"])
        loss = (xN * state["gx"]).sum() + (vN * state["gx"]).sum()
        return {"x": xN.detach(), "v": vN.detach(), "grads": list(torch.autograd.grad(loss, leaves))}
    s.calc_neighbor_list(state["cut"])
    s.calc_force_energy()
    return {"epot": s.potential_energy(), "phi": s.phi(), "fmax": s.max_unbalanced_force(), "force": _field(s, "force"),
            "area": _field(s, "area"), "perimeter": _field(s, "perimeter")}


def work(case):
    """State read and written once; per step, the arithmetic of the shape terms (about 120 operations a
    vertex), of the integrator and of the pairs in contact range (three a vertex: 25 operations for a
    vertex pair, 60 for a vertex on a segment).  A reverse pass does three times a step's arithmetic."""
    counts = _ring_counts(case)
    nv = sum(counts) * 0.5 * (case["n_small"] + case["n_large"])
    step = nv * (140 + 3 * (60 if case.get("inter") == "vertexSmooth" else 25))
    if case["kind"] == "rigid":
        return {"bytes": nv * 8 * 6 + sum(counts) * 8 * 12, "flops": case["steps"] * nv * (40 + 3 * 60)}
    if case["kind"] == "fire":
        return {"bytes": nv * 8 * 14, "flops": 2 * case["iters"] * step}
    if case["kind"] == "grad":
        return {"bytes": nv * 8 * 20, "flops": 4 * case["steps"] * step}
    if case["kind"] == "setup":
        return {"bytes": nv * 8 * 8 + nv * 6 * 4, "flops": step + nv * 60 * 10}
    return {"bytes": nv * 8 * 12, "flops": case["steps"] * step}


# ----------------------------------------------------------- the same in plain torch, 64 bits
class _Plain:
    """Energies of the packing in torch, forces by differentiation."""

    def __init__(self, case, p):
        self.case, self.p, self.q = case, p, _settings(case, p)
        box = torch.as_tensor(p["box"], device=DEV)
        self.sys = p["sys_of_ring"][p["ring"]]
        self.box = box[self.sys]
        self.nsys = len(p["counts"])
        self.rad, self.l0, self.a0 = p["rad"], p["l0"], p["a0"]
        self.n = torch.as_tensor(p["nvp"], device=DEV)
        ea, el, eb, self.ec = self.q["costs"]
        one = torch.ones(len(self.n), dtype=F64, device=DEV)
        self.ka, self.kl, self.kb = ea * one, el * one, eb * one
        self.smooth = case.get("inter") == "vertexSmooth"
        self.pot = case.get("pot", "harmonic")
        self.reach = {"harmonic": 1.0, "wca": KWCA, "adhesive": 1.2, "lj": 1.5}[self.pot]
        self.pairs(p["pos"])

    def im(self, d, b):
        return d - b * torch.round(d.detach() / b)

    def pairs(self, x):
        """Ordered pairs (i, j) of different rings that can come into range (for segments: i and the
        segment that ends in j), from the rings of the neighbouring lattice sites."""
        p = self.p
        most = int(self.n.max())
        k = torch.arange(most, device=DEV)
        slot = p["first"][:, None] + k[None]
        slot = torch.where(k[None] < self.n[:, None], slot, torch.full_like(slot, -1))
        got = []
        self.at = x.clone()
        for q in range(p["ring_nb"].shape[1]):
            nb = p["ring_nb"][:, q]
            for part in torch.arange(len(nb), device=DEV)[nb >= 0].split(4096):
                i = slot[part][:, :, None].expand(-1, -1, most)
                j = slot[nb[part]][:, None, :].expand(-1, most, -1)
                ok = (i >= 0) & (j >= 0)
                i, j = i[ok], j[ok]
                d = self.im(x[i] - x[j], self.box[i]).norm(dim=-1)
                sig = self.rad[i] + self.rad[j]
                near = d < (self.reach + 0.7 + (1.4 if self.smooth else 0.0)) * sig
                got.append(i[near] * x.shape[0] + j[near])
        key = torch.unique(torch.cat(got))
        i, j = key // x.shape[0], key % x.shape[0]
        if not self.smooth:
            i, j = i[i < j], j[i < j]
        self.i, self.j = i, j

    def V(self, d, sig):
        """The pair potential, zero beyond its reach."""
        if self.pot == "harmonic":
            e = 0.5 * self.ec * (1 - d / sig) ** 2
        elif self.pot == "adhesive":
            o, l1, l2 = 1 - d / sig, 0.1, 0.2
            e = torch.where(d < (1 + l1) * sig, 0.5 * self.ec * (o * o - l1 * l2), -0.5 * self.ec * l1 / (l2 - l1) * (o + l2) ** 2)
        else:
            s6 = (sig / d) ** 6
            e = 4 * self.ec * (s6 * s6 - s6)
            if self.pot == "wca":
                e = e + self.ec
            else:
                c6 = 1.5 ** -6
                cut = 4 * self.ec * (c6 * c6 - c6)
                shift = 24 * self.ec * (2 * c6 * c6 - c6) / 1.5 / sig
                e = e - cut - abs(shift) * (d - 1.5 * sig)
        return torch.where(d <= self.reach * sig, e, torch.zeros_like(e))

    def inter(self, x):
        i, j = self.i, self.j
        b, sig = self.box[i], self.rad[i] + self.rad[j]
        safe = lambda v: torch.sqrt((v * v).sum(-1))  # noqa: E731
        if not self.smooth:
            return self.V(safe(self.im(x[i] - x[j], b)), sig), self.sys[i]
        pj = self.p["prev"][j]
        qj = self.p["prev"][pj]
        sg, ip = self.im(x[j] - x[pj], b), self.im(x[i] - x[pj], b)
        ps, iq = self.im(x[qj] - x[pj], b), self.im(x[i] - x[qj], b)
        t = (ip * sg).sum(-1) / (sg * sg).sum(-1)
        u = -((iq * ps).sum(-1) / (ps * ps).sum(-1)).detach()
        on, corner = (t >= 0) & (t < 1), self.V(safe(ip), sig)
        wall = self.V(safe(ip - t.clamp(0, 1)[:, None] * sg), sig)
        zero = torch.zeros_like(wall)
        e = torch.where(on, wall - torch.where((u >= 0) & (u < 1), corner, zero), torch.where((t < 0) & (u >= 1), corner, zero))
        return e, self.sys[i]

    def geometry(self, x):
        p, ring = self.p, self.p["ring"]
        d = self.im(x[p["next"]] - x, self.box)
        cs = torch.cumsum(d, 0)
        f = p["first"]
        u = cs - d - (cs[f] - d[f])[ring]
        add = lambda v: torch.zeros(len(self.n), dtype=F64, device=DEV).index_add(0, ring, v)  # noqa: E731
        length = torch.sqrt((d * d).sum(-1))
        shoe = add(u[:, 0] * d[:, 1] - d[:, 0] * u[:, 1])
        # the turning angle, with the sign the engine gives it
        e = d[p["prev"]]
        theta = torch.atan2(d[:, 0] * e[:, 1] - d[:, 1] * e[:, 0], (d * e).sum(-1))
        centre = x.detach()[f] + torch.stack([add(u.detach()[:, k]) for k in (0, 1)], -1) / self.n[:, None]
        return 0.5 * shoe.abs(), length, theta, add(length.detach()), centre

    def shape(self, x):
        ring = self.p["ring"]
        area, length, theta, _, _ = self.geometry(x)
        e_ring = 0.5 * self.ka * (area / self.a0 - 1) ** 2
        e = 0.5 * self.kl[ring] * (length / self.l0 - 1) ** 2 + 0.5 * self.kb[ring] * (theta - self.p["theta0"]) ** 2
        return e_ring, e

    def energy(self, x, rigid=False):
        """Per-system potential energy."""
        e, s = self.inter(x)
        U = torch.zeros(self.nsys, dtype=F64, device=DEV).index_add(0, s, e)
        if rigid:
            return U
        er, ev = self.shape(x)
        return U.index_add(0, self.p["sys_of_ring"], er).index_add(0, self.sys, ev)

    def force(self, x, rigid=False, graph=False):
        if not graph:
            x = x.detach().requires_grad_()
        if ((x - self.at).detach().abs() > 0.15 * self.p["size"]).any():
            self.pairs(x.detach())
        return -torch.autograd.grad(self.energy(x, rigid).sum(), x, create_graph=graph)[0]

    def sum_sys(self, v):
        return torch.zeros(self.nsys, dtype=F64, device=DEV).index_add(0, self.sys, v)


def _philox(counter, index, tag, system, seed):
    """Philox4x32-10 on arrays: two Gaussians by Box and Muller."""
    u = lambda v: np.asarray(v, dtype=np.uint64)  # noqa: E731
    low, m32 = u(0xFFFFFFFF), u(32)
    c0, c1 = np.broadcast_arrays(u(index), u(counter) & low)
    c2, c3 = np.zeros_like(c0), np.broadcast_to((u(tag) << u(24)) | u(system), c0.shape)
    k0, k1 = u(seed) & low, u(seed) >> m32
    for r in range(10):
        if r:
            k0, k1 = (k0 + u(0x9E3779B9)) & low, (k1 + u(0xBB67AE85)) & low
        p0, p1 = u(0xD2511F53) * c0, u(0xCD9E8D57) * c2
        c0, c1, c2, c3 = (p1 >> m32) ^ c1 ^ k0, p1 & low, (p0 >> m32) ^ c3 ^ k1, p0 & low
    one = lambda hi, lo: (((hi << m32) | lo) >> u(11)).astype(np.float64) + 0.5  # noqa: E731
    a, b = one(c0, c1) / 2.0 ** 53, one(c2, c3) / 2.0 ** 53
    r = np.sqrt(-2 * np.log(a))
    return torch.as_tensor(np.stack([r * np.cos(2 * PI * b), r * np.sin(2 * PI * b)], -1), device=DEV)


def _exact_md(case, p, seed):
    e = _Plain(case, p)
    q, ring, noise = e.q, p["ring"], case["noise"]
    dt, g, T = q["dt"], q["gamma"], p["T"]
    h = 0.5 * dt
    index = np.concatenate([np.arange(c) for c in p["counts"]])
    sysr = p["sys_of_ring"].cpu().numpy()
    draw_ = lambda tag, call: _philox(call, index, tag, sysr, seed + 17)  # noqa: E731
    ang = p["angle"].clone()

    calls = [0]

    def total(x):
        f = e.force(x)
        if noise == "active":
            nonlocal ang
            calls[0] += 1
            ang = ang + math.sqrt(2 * dt / q["taup"]) * draw_(3, calls[0])[:, 0] + PI
            ang = ang - 2 * PI * torch.floor(ang / (2 * PI)) - PI
            f = f + q["driving"] * torch.stack([torch.cos(ang), torch.sin(ang)], -1)[ring]
        return f

    x, v = p["pos"].clone(), p["vel"].clone()
    if noise == "active":  # the force of the set-up: its own angles were all zero, one draw each
        a = math.sqrt(2 * dt / q["taup"]) * draw_(3, 0)[:, 0]
        f = e.force(x) + q["driving"] * torch.stack([torch.cos(a), torch.sin(a)], -1)[ring]
    else:
        f = e.force(x)
    amp = math.sqrt(2 * T * g / dt)
    for k in range(case["steps"]):
        z = None if noise == "nve" else draw_(1, k)[ring]
        if noise == "brownian":
            f = total(x)
            v = (f + amp * z) / g
            at, x = x, x + dt * v
            continue
        v = v + h * f
        if noise == "baoab":
            x = x + h * v
            v = math.exp(-g * dt) * v + math.sqrt(1 - math.exp(-2 * g * dt)) * math.sqrt(T) * z
            x = x + h * v
        else:
            x = x + dt * v
        f = total(x)
        if noise in ("langevin", "active"):
            f = f + amp * z - g * v
        v = v + h * f
        at = x
    out = {"epot": e.energy(at), "ekin": 0.5 * e.sum_sys((v * v).sum(-1)), "pos": list(x.t()), "vel": list(v.t()), "force": list(f.t())}
    if noise == "active":
        out["angle"] = ang
    return out


def _exact_rigid(case, p):
    e = _Plain(case, p)
    ring, dt = p["ring"], e.q["dt"]
    h = 0.5 * dt
    NR = len(e.n)
    add = lambda v: torch.zeros((NR,) + v.shape[1:], dtype=F64, device=DEV).index_add(0, ring, v)  # noqa: E731

    def load(x):
        c = e.geometry(x)[4]
        r, f = e.im(x - c[ring], e.box), e.force(x, rigid=True)
        return c, add(f), add(r[:, 0] * f[:, 1] - r[:, 1] * f[:, 0]) / add((r * r).sum(-1))

    x, w, ang = p["pos"].clone(), torch.zeros(NR, dtype=F64, device=DEV), torch.zeros(NR, dtype=F64, device=DEV)
    v = p["vel"][p["first"]].clone()
    c, F, tq = load(x)
    for _ in range(case["steps"]):
        v, w = v + h * F, w + h * tq
        r = e.im(x - c[ring], e.box)
        new, turn = c + dt * v, (dt * w)[ring]
        ang = ang + dt * w
        cs, sn = torch.cos(turn), torch.sin(turn)
        x = x + (new - c)[ring] + torch.stack([r[:, 0] * cs - r[:, 1] * sn, r[:, 0] * sn + r[:, 1] * cs], -1) - r
        c, F, tq = load(x)
        v, w = v + h * F, w + h * tq
    k = 0.5 * (v * v).sum(-1) + 0.5 * p["a0"] / PI * w * w
    ekin = torch.zeros(e.nsys, dtype=F64, device=DEV).index_add(0, p["sys_of_ring"], k)
    return {"ekin": ekin, "pos": list(x.t()), "pvel": list(v.t()), "omega": w, "pforce": list(F.t()), "angle": ang}


def _exact_fire(case, p):
    e = _Plain(case, p)
    a_start, f_dec, f_inc, f_a, dt0, dt_max, a_first = FIRE
    x, v = p["pos"].clone(), p["vel"].clone()
    box, sysr = torch.as_tensor(p["box"], device=DEV).prod(-1), p["sys_of_ring"]
    by = lambda s: s[e.sys][:, None]  # noqa: E731
    sizes = []
    for way in (1, -1):
        area, _, _, _, centre = e.geometry(x)
        if way == 1:
            r0 = e.rad[p["first"]]
            disks = area.detach() + PI * r0 * r0 * (0.5 * e.n - 1)
            phi = torch.zeros(e.nsys, dtype=F64, device=DEV).index_add(0, sysr, disks) / box
            grown = torch.sqrt((phi + DPHI) / phi)
        sc = grown if way == 1 else 1 / grown
        x = x + by(sc - 1) * (x - centre[p["ring"]])
        e.rad, e.l0, e.a0 = e.rad * sc[e.sys], e.l0 * sc[e.sys], e.a0 * sc[sysr] ** 2
        e.pairs(x)
        f = e.force(x)
        dt = torch.full((e.nsys,), dt0, dtype=F64, device=DEV)
        a, num = torch.full_like(dt, a_first), torch.zeros_like(dt)
        for _ in range(case["iters"]):
            up = e.sum_sys((v * f).sum(-1)) > 0
            num = torch.where(up, num + 1, torch.zeros_like(num))
            grow = up & (num > 20)
            dt = torch.where(grow, (dt * f_inc).clamp(max=dt_max), torch.where(up, dt, (dt * f_dec).clamp(min=dt_max / 10)))
            a = torch.where(grow, a * f_a, torch.where(up, a, torch.full_like(a, a_start)))
            x = torch.where(by(up), x, x - by(0.5 * dt) * v)
            v = torch.where(by(up), v, torch.zeros_like(v)) + by(0.5 * dt) * f
            vv, ff = e.sum_sys((v * v).sum(-1)), e.sum_sys((f * f).sum(-1))
            v = by(1 - a) * v + by(a) * f * by(torch.sqrt(vv / ff))
            x = x + by(dt) * v
            f = e.force(x)
            v = v + by(0.5 * dt) * f
        count = e.sum_sys(torch.ones_like(e.rad))
        sizes.append(torch.sqrt(e.sum_sys((f * f).sum(-1)) / (2 * count)))
    return {"force_size": sizes, "epot": e.energy(x), "pos": list(x.t()), "vel": list(v.t()), "force": list(f.t()), "l0": e.l0}


def _exact_grad(case, p):
    e = _Plain(case, p)
    leaves = [t.clone().requires_grad_() for t in (p["pos"].reshape(-1), p["vel"].reshape(-1), e.ka, e.kl, e.kb, p["l0"])]
    x, v, e.ka, e.kl, e.kb, e.l0 = leaves
    x, v, dt = x.reshape(-1, 2), v.reshape(-1, 2), e.q["dt"]
    f = e.force(x, graph=True)
    for _ in range(case["steps"]):
        v = v + 0.5 * dt * f
        x = x + dt * v
        f = e.force(x, graph=True)
        v = v + 0.5 * dt * f
    x, v = x.reshape(-1), v.reshape(-1)
    loss = (x * p["grad_x"]).sum() + (v * p["grad_x"]).sum()
    return {"x": x.detach(), "v": v.detach(), "grads": list(torch.autograd.grad(loss, leaves))}


def exact(case, seed):
    p = packing(case, seed)
    if case["kind"] == "md":
        return _exact_md(case, p, seed)
    if case["kind"] == "rigid":
        return _exact_rigid(case, p)
    if case["kind"] == "fire":
        return _exact_fire(case, p)
    if case["kind"] == "grad":
        return _exact_grad(case, p)
    e = _Plain(case, p)
    area, _, _, perimeter, _ = e.geometry(p["pos"])
    f = e.force(p["pos"])
    r0 = e.rad[p["first"]]
    disks = area + PI * r0 * r0 * (0.5 * e.n - 1)
    phi = torch.zeros(e.nsys, dtype=F64, device=DEV).index_add(0, p["sys_of_ring"], disks)
    top = torch.zeros(e.nsys, dtype=F64, device=DEV).scatter_reduce(0, e.sys, f.abs().max(-1).values, "amax")
    return {"epot": e.energy(p["pos"]), "phi": phi / torch.as_tensor(p["box"], device=DEV).prod(-1), "fmax": top, "force": list(f.t()),
            "area": area, "perimeter": perimeter}
