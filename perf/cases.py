"""The work whose speed counts: cases a program hands to this package's
public entry points (Simulation, FrameEvaluator, frame_forces),
over the range of sizes and options they are used at.

listed() names fixed cases, draw(rng) makes more of the same ranges,
prepare() builds what a program holds before the call, run() is one pass,
exact() the same pass in 64 bits in plain torch (cell-free pair lists, PME
on torch.fft, constraints by Newton iteration, derivatives by autograd).

Boxes come from a small periodic box (a "unit"), relaxed here by a few
descent steps, repeated along x, y and z: a large box is built from a
relaxed small one, and the velocities differ from copy to copy.
"""
from __future__ import annotations

import dataclasses
import itertools
import math

import numpy as np
import torch

# torch's HIP runtime has to be up before the library loads
from mdir_amd.torch_frames import frame_forces
from mdir_amd import systems as S
from mdir_amd.frames import FrameEvaluator
from mdir_amd.simulation import Simulation

F64 = torch.float64
DEV = "cuda"
COULOMB = 138.93545755023302   # kJ nm mol^-1 e^-2
KB = 0.008314462618153241      # kJ mol^-1 K^-1
DT = 0.002                     # ps


# ---- the cases ----------------------------------------------------------------

def listed():
    return [
        # The smallest run: liquid argon, 864 atoms, no charges, where a step
        # is launches and latency.
        _md("argon_864_nve", "argon", 0, (6, 6, 6), steps=50, skin=0.1),
        # A small solvated box (the smallest replica size), alone on the GPU.
        _md("water_500_nve", "water", 500, (1, 1, 1), steps=50, spacing=0.12, skin=0.15),
        # The ordinary production run: the ~24k-atom PME water box.
        _md("water_24k_nve", "water", 988, (2, 2, 2), steps=50, skin=0.2),
        # A ragged, non-cubic box with order-6 splines under Langevin dynamics.
        _md("water_14k_order6_langevin", "water", 777, (3, 2, 1), steps=50, order=6,
            spacing=0.12, skin=0.15, langevin=True),
        # Solutes with bonded terms, constrained bonds and a force switch.
        _md("solutes_25k_bonded_langevin", "solutes", 1000, (2, 2, 2), steps=50, switch=0.7,
            skin=0.15, langevin=True),
        # A larger solvated system of about a hundred thousand atoms.
        _md("water_107k_nve", "water", 988, (3, 4, 3), steps=20, skin=0.15),
        # The largest: a million atoms under Langevin with volume moves.
        _md("water_999k_npt", "water", 971, (7, 7, 7), steps=50, skin=0.15, langevin=True,
            npt=True),
        # One evaluation at new positions (rescoring, minimisers, path
        # methods): list build, forces and every energy term to the host.
        dict(_md("water_24k_forces", "water", 988, (2, 2, 2), steps=0, skin=0.1), kind="forces"),
        # Force matching: 64 frames of 3,150 atoms per call, arrays on the GPU.
        _frames("frames_64_force_matching", "matching", 64, 1000),
        # The same for one frame per call, where launches count.
        _frames("frames_1_force_matching", "matching", 1, 1000),
        # Energies and forces inside a torch program, differentiated through:
        # forward, then gradients in positions and parameters.
        _frames("frames_8_autograd", "autograd", 8, 1000),
    ]


def _md(name, system, unit, tiles, steps, order=4, spacing=0.1, skin=0.1, switch=0.0,
        langevin=False, npt=False):
    return {"name": name, "kind": "md", "system": system, "unit": unit, "tx": tiles[0],
            "ty": tiles[1], "tz": tiles[2], "steps": steps, "order": order, "spacing": spacing,
            "skin": skin, "switch": switch, "langevin": langevin, "npt": npt}


def _frames(name, kind, count, unit):
    return {"name": name, "kind": kind, "count": count, "unit": unit}


def draw(rng):
    """One more case: sizes uniform in their logarithm over the listed range."""
    kind = rng.choice(["md", "md", "md", "forces", "matching", "matching", "autograd"])
    if kind in ("matching", "autograd"):
        most = 64 if kind == "matching" else 12
        count = max(1, min(most, int(math.exp(rng.uniform(0.0, math.log(most + 0.99))))))
        c = _frames("", kind, count, rng.randint(600, 1000))
    else:
        total = math.exp(rng.uniform(math.log(500), math.log(330000 if kind == "md" else 36000)))
        if kind == "md" and total < 3000 and rng.random() < 0.3:
            c = _md("", "argon", 0, tuple(rng.randint(5, 9) for _ in range(3)), steps=50,
                    skin=rng.choice([0.1, 0.15]))
        else:
            unit = rng.randint(500, 988)
            copies = max(1, round(total / unit))
            tx = max(1, min(copies, round(copies ** (1 / 3) * rng.uniform(0.8, 1.25))))
            ty = max(1, min(copies // tx, round(math.sqrt(copies / tx) * rng.uniform(0.8, 1.25))))
            tz = max(1, copies // (tx * ty))
            solutes = unit >= 600 and copies <= 36 and rng.random() < 0.3
            steps = 50 if copies < 40 else 20
            c = _md("", "solutes" if solutes else "water", unit, (tx, ty, tz), steps=steps,
                    order=rng.choice([4, 4, 4, 6]), spacing=rng.choice([0.1, 0.12]),
                    skin=rng.choice([0.1, 0.15, 0.2]) if unit >= 560 else 0.1,
                    switch=0.7 if solutes else 0.0, langevin=rng.random() < 0.5)
            if kind == "forces":
                c.update(kind="forces", steps=0, langevin=False)
    del c["name"]
    return c


# ---- inputs -------------------------------------------------------------------

@dataclasses.dataclass
class Inputs:
    """A System (host arrays) and the velocities its run starts from."""
    system: S.System
    velocities: np.ndarray


def _unit(case, seed):
    """The relaxed small box the case's box repeats."""
    if case["system"] == "water":
        n = case["unit"]
        s = S.tip3p_box(n, S.water_edge(n, 0.995), seed=seed, grid=(16, 16, 16))
    else:
        s = _solutes(case["unit"], seed)
        if case["switch"]:
            s = dataclasses.replace(s, lj_modifier=S.LJ_FORCE_SWITCH, switch_from=case["switch"])
    return dataclasses.replace(s, positions=_relax(s))


def _solutes(waters, seed):
    """Water with five-site solutes bound to their centre: every second one
    with bonds of fixed length, the others with springs; angles at the
    centre in all of them."""
    solutes = max(2, (3 * waters) // 100)
    s = S.solvated_solutes(waters, solutes, seed=seed)
    first = 3 * waters + 5 * np.arange(solutes)
    pairs = np.stack([np.stack([first, first + k], 1) for k in range(1, 5)], 1)
    angles = np.concatenate([np.stack([first + a, first, first + b], 1)
                             for a, b in itertools.combinations(range(1, 5), 2)])
    stiff, loose = pairs[0::2].reshape(-1, 2), pairs[1::2].reshape(-1, 2)
    return dataclasses.replace(
        s, constraints=stiff.astype(np.int32), constraint_length=np.full(len(stiff), 0.1),
        bonds=loose.astype(np.int32), bond_k=np.full(len(loose), 150000.0),
        bond_r0=np.full(len(loose), 0.1), angles=angles.astype(np.int32),
        angle_k=np.full(len(angles), 400.0),
        angle_theta0=np.full(len(angles), math.acos(-1.0 / 3.0)))


def _tile(s, tiles, spacing, order):
    """`s` repeated along x, y and z, with the PME grid of the whole box."""
    cells = np.array(list(itertools.product(*(range(t) for t in tiles))))
    m, n = len(cells), s.n
    first = np.arange(m) * n

    def atoms(a):
        a = np.asarray(a)
        return (a[None] + first.reshape((-1,) + (1,) * a.ndim)).reshape((-1,) + a.shape[1:]) \
            .astype(np.int32)

    def rep(a):
        a = np.asarray(a)
        return np.tile(a, (m,) + (1,) * (a.ndim - 1))

    box = s.box * np.asarray(tiles)
    x = (s.positions[None] + (cells * s.box)[:, None]).reshape(-1, 3)
    grid = S.pme_grid(box, spacing) if s.beta > 0 else (0, 0, 0)
    return dataclasses.replace(
        s, positions=x, box=box, masses=rep(s.masses), charges=rep(s.charges),
        types=rep(s.types), exclusions=atoms(s.exclusions), waters=atoms(s.waters),
        constraints=atoms(s.constraints), constraint_length=rep(s.constraint_length),
        bonds=atoms(s.bonds), bond_k=rep(s.bond_k), bond_r0=rep(s.bond_r0),
        angles=atoms(s.angles), angle_k=rep(s.angle_k), angle_theta0=rep(s.angle_theta0),
        pme_grid=grid, pme_order=order)


def _inputs(case, seed):
    tiles = (case["tx"], case["ty"], case["tz"])
    if case["system"] == "argon":
        cells = np.array(list(itertools.product(*(range(t) for t in tiles))), np.float64)
        basis = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]]) + 0.25
        x = ((cells[:, None] + basis) * (3.47 / 6)).reshape(-1, 3)
        one = S.argon_config1()
        s = dataclasses.replace(one, positions=x, masses=np.full(len(x), 39.95),
                                charges=np.zeros(len(x)), types=np.zeros(len(x), np.int32),
                                box=np.array(tiles) * (3.47 / 6),
                                exclusions=np.zeros((0, 2), np.int32))
        temperature = 120.0
    else:
        s = _tile(_unit(case, seed), tiles, case["spacing"], case["order"])
        temperature = 300.0
    return Inputs(s, _velocities(s, seed, temperature))


def _frame_inputs(case, seed):
    """The system of a frame batch, its frames (moves of 0.01 nm and 0.1 rad
    of every molecule and solute atom), reference forces or cotangents."""
    unit = case["unit"]
    s = S.solvated_solutes(unit, max(2, (3 * unit) // 100), seed=seed)
    s = dataclasses.replace(s, pme_grid=S.pme_grid(s.box, 0.1))
    s = dataclasses.replace(s, positions=_relax(s))
    gen = torch.Generator("cpu").manual_seed(seed)
    k, n = case["count"], s.n
    x0 = torch.from_numpy(s.positions)
    w = torch.from_numpy(s.waters.astype(np.int64))
    x = x0 + 0.01 * torch.randn((k, n, 3), generator=gen, dtype=F64)
    turn = 0.1 * torch.randn((k, len(w), 3), generator=gen, dtype=F64)
    angle = turn.norm(dim=-1, keepdim=True)
    axis = turn / angle
    for a in (1, 2):
        r = (x0[w + a] - x0[w]).expand(k, -1, 3)
        x[:, w + a] = x[:, w] + r * angle.cos() + torch.linalg.cross(axis, r) * angle.sin() + \
            axis * (axis * r).sum(-1, keepdim=True) * (1 - angle.cos())
    return s, x.to(DEV), gen


# ---- prepare and run ------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("md", "forces"):
        inp = _inputs(case, seed)
        sim = Simulation(inp.system, skin=case["skin"])
        sim.velocities = inp.velocities
        if case["langevin"]:
            sim.set_langevin(300.0, 1.0, seed=seed)
        state = {"case": case, "seed": seed, "sim": sim}
        if kind == "forces":
            state["x"] = _moved(inp.system, seed)
        return state
    s, x, gen = _frame_inputs(case, seed)
    ev = FrameEvaluator(s, max_frames=case["count"])
    theta = ev.tunables
    state = {"case": case, "ev": ev, "x": x}
    if kind == "matching":
        state["ref"] = _reference_forces(s, x, seed)
    else:
        for name in ("charges", "sigma", "epsilon"):
            state[name] = torch.from_numpy(theta[name]).to(DEV).requires_grad_()
        x.requires_grad_()
        state["ge"], state["gf"] = _cotangents(case, x, gen)
    return state


def _reference_forces(s, x, seed):
    """Forces of the frames at parameters moved by up to 2 %."""
    q, sig, eps = S.perturbed_parameters(s, seed=seed % 100000)
    box = torch.tensor(s.box, dtype=F64, device=DEV)
    top = _Topology(S.with_parameters(s, q, sig, eps))
    return torch.stack([top.forces(xk, box)[0] for xk in x])


def _cotangents(case, x, gen):
    ge = torch.randn(case["count"], generator=gen, dtype=F64).to(DEV)
    gf = 0.01 * torch.randn(tuple(x.shape), generator=gen, dtype=F64).to(DEV)
    return ge, gf


def _moved(s, seed):
    """Positions to rescore: every molecule of the box shifted a little."""
    rng = np.random.default_rng(seed + 1)
    x = s.positions.copy()
    shift = rng.normal(0.0, 0.005, (len(s.waters), 3))
    for k in range(3):
        x[s.waters + k] += shift
    return x


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "md":
        sim = state["sim"]
        if case["npt"]:
            ke = sim.run_npt(case["steps"], DT, graph=50, every=case["steps"], pressure=1.0,
                             temperature=300.0, seed=state["seed"])
        else:
            ke = sim.run(case["steps"], DT, graph=50)
        out = {"positions": sim.positions, "velocities": sim.velocities, "kinetic": ke}
        if case["npt"]:
            out["box"] = sim.box
        return out
    if kind == "forces":
        sim = state["sim"]
        sim.positions = state["x"]
        forces, energies = sim.forces()
        return {"forces": forces, "energies": energies}
    ev = state["ev"]
    if kind == "matching":
        loss, grad = ev.force_matching(state["x"], state["ref"])
        return {"loss": loss, **{k: grad[k] for k in ("charges", "sigma", "epsilon")}}
    inputs = [state["x"]] + [state[k] for k in ("charges", "sigma", "epsilon")]
    energy, forces = frame_forces(ev, *inputs)
    loss = (state["ge"] * energy).sum() + (state["gf"] * forces).sum()
    dx, dq, ds, de = torch.autograd.grad(loss, inputs)
    return {"energy": energy.detach(), "forces": forces.detach(), "positions": dx,
            "charges": dq, "sigma": ds, "epsilon": de}


# ---- work and tolerance -----------------------------------------------------------

def _sizes(case):
    """(atoms, box volume, PME points) of one box of the case."""
    if case["system"] == "argon":
        cells = case["tx"] * case["ty"] * case["tz"]
        return 4 * cells, cells * (3.47 / 6) ** 3, 0
    copies = case["tx"] * case["ty"] * case["tz"]
    edge = S.water_edge(case["unit"], 0.995)
    atoms = 3 * case["unit"]
    if case["system"] == "solutes":
        solutes = max(2, (3 * case["unit"]) // 100)
        atoms += 5 * solutes
        edge = (S.water_edge(case["unit"]) ** 3 + 0.1 * solutes) ** (1 / 3)
    grid = S.pme_grid([edge * t for t in (case["tx"], case["ty"], case["tz"])], case["spacing"])
    return atoms * copies, edge ** 3 * copies, int(np.prod(grid))


def _force_flops(atoms, volume, points, order):
    """Pairs inside the cutoff (50 operations each), spread and gather (6 a
    stencil point) and two real transforms of one evaluation."""
    rc = 1.0 if points == 0 else 0.9
    pairs = 0.5 * atoms * atoms / volume * 4.0 / 3.0 * math.pi * rc ** 3
    flops = 50.0 * pairs
    if points:
        flops += 2 * 6 * atoms * order ** 3 + 5.0 * points * math.log2(points)
    return flops


def work(case):
    """Positions and velocities are read and written once a step (a state of
    48 bytes an atom); a force evaluation reads positions and writes forces;
    a gradient call reads frames and reference forces."""
    kind = case["kind"]
    if kind in ("matching", "autograd"):
        unit = case["unit"]
        sol = max(2, (3 * unit) // 100)
        atoms, volume = 3 * unit + 5 * sol, S.water_edge(unit) ** 3 + 0.1 * sol
        points = 32 ** 3
        per = _force_flops(atoms, volume, points, 4)
        passes = 2.0 if kind == "matching" else 4.0
        frame = 48.0 if kind == "matching" else 96.0
        return {"bytes": case["count"] * atoms * frame, "flops": case["count"] * passes * per}
    atoms, volume, points = _sizes(case)
    per = _force_flops(atoms, volume, points, case["order"])
    if kind == "forces":
        return {"bytes": 48.0 * atoms, "flops": per}
    evaluations = case["steps"] + (2 if case["npt"] else 0)
    return {"bytes": 96.0 * atoms * case["steps"], "flops": per * evaluations}


def tolerance(case):
    """f32 pair and mesh arithmetic, four times the errors seen against 64
    bits: 2.5e-6 of the forces of one evaluation, 5e-6 of force-matching
    gradients, 2e-6 of the autograd's.  A run carries the force error along
    its steps (velocities: 1e-5 after 50 steps, 1e-4 after 100)."""
    kind = case["kind"]
    if kind == "matching":
        return {"rel": 2e-5, "max": 1e-3}
    if kind in ("forces", "autograd"):
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 4e-4, "max": 0.05}


# ---- the same in 64 bits, in plain torch ----------------------------------------------

def _t(a, dtype=F64):
    return torch.as_tensor(np.asarray(a), dtype=dtype, device=DEV)


def _spline(w, order):
    """B-spline weights of the points floor(u) - order + 1 + t."""
    a = [w, 1.0 - w]
    for n in range(3, order + 1):
        b = a + [torch.zeros_like(w)]
        a = [((w + k) * b[k] + ((n - w - k) * b[k - 1] if k else 0.0)) / (n - 1) for k in range(n)]
    return torch.stack(a[::-1], -1)


class _Topology:
    """A System's force field in 64 bits: energies of positions, and what
    autograd makes of them."""

    def __init__(self, s):
        self.s = s
        self.q = _t(s.charges)
        self.types = _t(s.types, torch.int64)
        self.sigma, self.eps = _t(s.sigma), _t(s.epsilon)
        ex = _t(s.exclusions.reshape(-1, 2), torch.int64)
        self.ex_i, self.ex_j = ex[:, 0], ex[:, 1]
        self.keys = torch.sort(self.ex_i * s.n + self.ex_j).values
        self.mass = _t(s.masses)
        self.list = None

    def pairs(self, x, box, reach):
        """The non-excluded pairs within `reach`."""
        n, out = len(x), []
        rows = max(1, min(n, 50_000_000 // n))
        for a in range(0, n, rows):
            i = torch.arange(a, min(a + rows, n), device=DEV)
            r2 = torch.zeros((len(i), n - a), dtype=F64, device=DEV)
            for k in range(3):
                d = x[a:, k][None] - x[i, k][:, None]
                d -= box[k] * torch.round(d / box[k])
                r2 += d * d
            hit = torch.nonzero(r2 < reach * reach)
            pi, pj = hit[:, 0] + a, hit[:, 1] + a
            keep = pj > pi
            out.append(torch.stack([pi[keep], pj[keep]]))
        p = torch.cat(out, 1)
        if len(self.keys):
            key = p[0] * n + p[1]
            at = torch.searchsorted(self.keys, key).clamp(max=len(self.keys) - 1)
            p = p[:, self.keys[at] != key]
        return p

    def energy(self, x, box, pairs, q=None, sigma=None, eps=None):
        """Energy terms by name (sigma, eps per type: Lorentz-Berthelot)."""
        s = self.s
        q = self.q if q is None else q
        out = {}

        def between(i, j):
            d = x[j] - x[i]
            return d - box * torch.round(d.detach() / box.detach())

        i, j = pairs
        d = between(i, j)
        r2 = (d * d).sum(-1)
        near = torch.nonzero(r2 < s.cutoff ** 2)[:, 0]
        i, j, r2 = i[near], j[near], r2[near]
        ti, tj = self.types[i], self.types[j]
        lj = torch.nonzero(self.eps[ti, tj] > 0)[:, 0]
        ti, tj, l2 = ti[lj], tj[lj], r2[lj]
        if sigma is None:
            sg, ep = self.sigma[ti, tj], self.eps[ti, tj]
        else:
            sg, ep = 0.5 * (sigma[ti] + sigma[tj]), torch.sqrt(eps[ti] * eps[tj])
        s6 = sg ** 6
        i6 = l2 ** -3
        p12 = p6 = 0.0
        if s.lj_modifier == S.LJ_FORCE_SWITCH:
            u = (l2.sqrt() - s.switch_from).clamp(min=0.0)
            p12, p6 = (self._switch(m, u) for m in (12.0, 6.0))
        out["lj"] = (4 * ep * (s6 * s6 * (i6 * i6 - p12) - s6 * (i6 - p6))).sum()
        if s.beta > 0:
            r = r2.sqrt()
            out["direct"] = (COULOMB * q[i] * q[j] * torch.erfc(s.beta * r) / r).sum()
            de = between(self.ex_i, self.ex_j)
            re = (de * de).sum(-1).sqrt()
            out["excluded"] = -(COULOMB * q[self.ex_i] * q[self.ex_j] *
                                torch.erf(s.beta * re) / re).sum()
            out["recip"] = self._mesh(x, box, q)
            out["self"] = -COULOMB * s.beta / math.sqrt(math.pi) * (q * q).sum() - \
                COULOMB * math.pi * q.sum() ** 2 / (2 * box.prod() * s.beta ** 2)
        if len(s.bonds):
            b = _t(s.bonds, torch.int64)
            db = between(b[:, 0], b[:, 1])
            out["bonds"] = (0.5 * _t(s.bond_k) * ((db * db).sum(-1).sqrt() - _t(s.bond_r0)) ** 2
                            ).sum()
        if len(s.angles):
            a = _t(s.angles, torch.int64)
            u, v = between(a[:, 1], a[:, 0]), between(a[:, 1], a[:, 2])
            th = torch.atan2(torch.linalg.cross(u, v).norm(dim=-1), (u * v).sum(-1))
            out["angles"] = (0.5 * _t(s.angle_k) * (th - _t(s.angle_theta0)) ** 2).sum()
        return out

    def _switch(self, n, u):
        rc, rs = self.s.cutoff, self.s.switch_from
        w = rc - rs
        a = -n * ((n + 4) * rc - (n + 1) * rs) / (rc ** (n + 2) * w ** 2)
        b = n * ((n + 3) * rc - (n + 1) * rs) / (rc ** (n + 2) * w ** 3)
        return rc ** -n - a / 3 * w ** 3 - b / 4 * w ** 4 + u ** 3 * (a / 3 + b / 4 * u)

    def _mesh(self, x, box, q):
        """The PME reciprocal energy."""
        s = self.s
        n, K = s.pme_order, s.pme_grid
        at, weight = [], []
        for a in range(3):
            u = x[:, a] / box[a]
            u = K[a] * (u - torch.floor(u.detach()))
            f = torch.floor(u.detach())
            weight.append(_spline(u - f, n))
            at.append((f.long()[:, None] - n + 1 + torch.arange(n, device=DEV)) % K[a])
        w = q[:, None, None, None] * weight[0][:, :, None, None] * weight[1][:, None, :, None] * \
            weight[2][:, None, None, :]
        idx = (at[0][:, :, None, None] * K[1] + at[1][:, None, :, None]) * K[2] + \
            at[2][:, None, None, :]
        grid = torch.zeros(K[0] * K[1] * K[2], dtype=F64, device=DEV)
        grid = grid.index_add(0, idx.reshape(-1), w.reshape(-1)).reshape(K)
        spec = torch.fft.rfftn(grid)
        node = _spline(torch.zeros((), dtype=F64, device=DEV), n).flip(0)[1:]
        m, mod = [], []
        for a in range(3):
            k = torch.arange(K[a], dtype=F64, device=DEV)
            ph = torch.exp(2j * math.pi * k[:, None] / K[a] *
                           torch.arange(n - 1, device=DEV)[None])
            mod.append(1.0 / (ph * node).sum(1).abs() ** 2)
            m.append(torch.where(k <= K[a] // 2, k, k - K[a]) / box[a])
        h = K[2] // 2 + 1
        m2 = m[0][:, None, None] ** 2 + m[1][None, :, None] ** 2 + m[2][None, None, :h] ** 2
        m2 = torch.where(m2 == 0, torch.full_like(m2, 1e30), m2)
        t = torch.exp(-math.pi ** 2 / s.beta ** 2 * m2) / m2 * mod[0][:, None, None] * \
            mod[1][None, :, None] * mod[2][None, None, :h]
        t = t * (COULOMB / (math.pi * box.prod()))
        half = torch.ones(h, dtype=F64, device=DEV)
        half[0] = 0.5
        if K[2] % 2 == 0:
            half[-1] = 0.5
        return (t * half * (spec.real ** 2 + spec.imag ** 2)).sum()

    def forces(self, x, box, pairs=None):
        if pairs is None:
            pairs = self.pairs(x, box, self.s.cutoff)
        x = x.detach().requires_grad_()
        terms = self.energy(x, box, pairs)
        return -torch.autograd.grad(sum(terms.values()), x)[0], \
            {k: float(v.detach()) for k, v in terms.items()}


class _Rigid:
    """The constraints of a system: rigid waters and fixed-length bonds to a
    centre, solved together per molecule by Newton steps."""

    def __init__(self, s):
        self.groups = []
        im = 1.0 / _t(s.masses)
        if len(s.waters):
            w = _t(s.waters, torch.int64)
            d = torch.tensor([s.water_geometry[0], s.water_geometry[0], s.water_geometry[1]],
                             dtype=F64, device=DEV)
            self._add(im, torch.stack([w, w + 1, w + 2], 1), [(0, 1), (0, 2), (1, 2)],
                      d.expand(len(w), 3))
        if len(s.constraints):
            c = s.constraints.reshape(-1, 4, 2)  # four bonds to one centre
            at = np.concatenate([c[:, :1, 0], c[:, :, 1]], 1)
            self._add(im, _t(at, torch.int64), [(0, k) for k in range(1, 5)],
                      _t(s.constraint_length.reshape(-1, 4)))

    def _add(self, im, at, bonds, length):
        inc = torch.zeros((len(bonds), at.shape[1]), dtype=F64, device=DEV)
        for b, (i, j) in enumerate(bonds):
            inc[b, i], inc[b, j] = -1.0, 1.0
        w = im[at]
        couple = torch.einsum("ka,ua,la->ukl", inc, w, inc)
        self.groups.append((at, inc, w, couple, length))

    @staticmethod
    def _solve(A, b):
        m = b.shape[-1]
        A = [[A[:, r, c] for c in range(m)] for r in range(m)]
        b = [b[:, r] for r in range(m)]
        for i in range(m):
            for r in range(i + 1, m):
                f = A[r][i] / A[i][i]
                for c in range(i, m):
                    A[r][c] = A[r][c] - f * A[i][c]
                b[r] = b[r] - f * b[i]
        for i in reversed(range(m)):
            for c in range(i + 1, m):
                b[i] = b[i] - A[i][c] * b[c]
            b[i] = b[i] / A[i][i]
        return torch.stack(b, -1)

    def positions(self, x0, x1, sweeps=10):
        x1 = x1.clone()
        for at, inc, w, couple, length in self.groups:
            s = torch.matmul(inc, x0[at])
            y = x1[at]
            for _ in range(sweeps):
                r = torch.matmul(inc, y)
                A = 2.0 * couple * (r[:, :, None] * s[:, None]).sum(-1)
                lam = self._solve(A, length ** 2 - (r * r).sum(-1))
                y = y + w[..., None] * torch.matmul(inc.T, lam[..., None] * s)
            x1[at] = y
        return x1

    def velocities(self, x, v):
        v = v.clone()
        for at, inc, w, couple, _ in self.groups:
            r = torch.matmul(inc, x[at])
            u = v[at]
            A = couple * (r[:, :, None] * r[:, None]).sum(-1)
            mu = self._solve(A, -(r * torch.matmul(inc, u)).sum(-1))
            v[at] = u + w[..., None] * torch.matmul(inc.T, mu[..., None] * r)
        return v


def _relax(s, steps=100):
    """Positions after descent steps of at most 0.01 nm of the waters (other
    atoms are held), in the pair forces alone, over all pairs: sums in a
    fixed order, so a seed gives one box."""
    rigid, box, x = _Rigid(dataclasses.replace(s, constraints=s.constraints[:0])), _t(s.box), \
        _t(s.positions)
    types, q = _t(s.types, torch.int64), _t(s.charges)
    c6 = (4 * _t(s.epsilon) * _t(s.sigma) ** 6)[types][:, types]
    c12 = (4 * _t(s.epsilon) * _t(s.sigma) ** 12)[types][:, types]
    qq = COULOMB * q[:, None] * q[None]
    off = torch.eye(s.n, dtype=torch.bool, device=DEV)
    ex = _t(s.exclusions, torch.int64)
    off[ex[:, 0], ex[:, 1]] = True
    off[ex[:, 1], ex[:, 0]] = True
    held = torch.ones(s.n, dtype=torch.bool, device=DEV)
    for k in range(3):
        held[_t(s.waters, torch.int64) + k] = False
    x = rigid.positions(x, x)
    for k in range(steps):
        d = x[None] - x[:, None]
        d -= box * torch.round(d / box)
        r2 = (d * d).sum(-1).masked_fill_(off, 1e30)
        r, i2 = r2.sqrt(), 1.0 / r2
        i6 = i2 ** 3
        fs = (12 * c12 * i6 - 6 * c6) * i6 + qq * (
            torch.erfc(s.beta * r) / r +
            2 * s.beta / math.sqrt(math.pi) * torch.exp(-s.beta ** 2 * r2))
        fs = torch.where(r2 < s.cutoff ** 2, fs * i2, torch.zeros_like(fs))
        f = -(fs[..., None] * d).sum(1)
        f[held] = 0.0
        f = f * (0.01 * 0.98 ** k / f.norm(dim=-1).max())
        x = rigid.positions(x, x + f, sweeps=4)
    return rigid.positions(x, x).cpu().numpy()


def _velocities(s, seed, temperature):
    """Maxwell-Boltzmann velocities that keep the constraints."""
    gen = torch.Generator(DEV).manual_seed(seed)
    m = _t(s.masses)[:, None]
    v = torch.randn((s.n, 3), generator=gen, dtype=F64, device=DEV) * torch.sqrt(KB * temperature / m)
    v = _Rigid(s).velocities(_t(s.positions), v)
    v = v - (m * v).sum(0) / m.sum()
    kinetic = 0.5 * (m * v * v).sum()
    return (v * torch.sqrt(0.5 * s.degrees_of_freedom() * KB * temperature / kinetic)).cpu().numpy()


def _philox(counter, key):
    """Philox 4x32-10 (Salmon et al., SC11) of uint64 arrays of 32-bit words."""
    c, low = [np.asarray(w, np.uint64) for w in counter], np.uint64(0xFFFFFFFF)
    k0, k1 = (np.uint64(k) for k in key)
    for _ in range(10):
        a, b = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(b >> np.uint64(32)) ^ c[1] ^ k0, b & low, (a >> np.uint64(32)) ^ c[3] ^ k1, a & low]
        k0, k1 = (k0 + np.uint64(0x9E3779B9)) & low, (k1 + np.uint64(0xBB67AE85)) & low
    return c


def _normals(seed, step, n):
    zero = np.zeros(n, np.uint64)
    w = _philox((zero + np.uint64(step), zero, np.arange(n, dtype=np.uint64),
                 zero + np.uint64(2 << 24)), (seed & 0xFFFFFFFF, seed >> 32))
    u = [(x.astype(np.float64) + 0.5) * 2.0 ** -32 for x in w]
    a, b = np.sqrt(-2 * np.log(u[0])), np.sqrt(-2 * np.log(u[2]))
    p = 2 * math.pi
    return _t(np.stack([a * np.cos(p * u[1]), a * np.sin(p * u[1]), b * np.cos(p * u[3])], 1))


def _dynamics(inp, case, seed):
    """`steps` steps of velocity Verlet or of geodesic BAOAB, then under NPT
    one volume move."""
    s = inp.system
    top, rigid, box = _Topology(s), _Rigid(s), _t(s.box)
    x, v, im = _t(s.positions), _t(inp.velocities), 1.0 / _t(s.masses)[:, None]
    decay = math.exp(-1.0 * DT)
    width = torch.sqrt((1 - decay ** 2) * KB * 300.0 * im)

    def drift(x, v, h):
        free = x + h * v
        new = rigid.positions(x, free)
        return new, v + (new - free) / h

    f = top.forces(x, box)[0]
    for step in range(case["steps"]):
        v = v + 0.5 * DT * im * f
        if case["langevin"]:
            v = rigid.velocities(x, v)
            x, v = drift(x, v, 0.5 * DT)
            v = rigid.velocities(x, decay * v + width * _normals(seed, step, s.n))
            x, v = drift(x, v, 0.5 * DT)
        else:
            x, v = drift(x, v, DT)
        if step % 10 == 0:
            pairs = top.pairs(x, box, s.cutoff + 0.12)
        f = top.forces(x, box, pairs)[0]
        v = rigid.velocities(x, v + 0.5 * DT * im * f)
    kinetic = 0.5 * float((v * v / im).sum())
    return x, v, kinetic


def exact(case, seed):
    kind = case["kind"]
    if kind == "md":
        if case["npt"] or _sizes(case)[0] * case["steps"] > 2.6e6:
            return None  # too long in plain torch
        x, v, kinetic = _dynamics(_inputs(case, seed), case, seed)
        return {"positions": x, "velocities": v, "kinetic": kinetic}
    if kind == "forces":
        inp = _inputs(case, seed)
        s = inp.system
        f, e = _Topology(s).forces(_t(_moved(s, seed)), _t(s.box))
        terms = [e["lj"], e["direct"], e["excluded"], e["recip"], e["self"], 0.0, 0.0, 0.0,
                 0.5 * float((s.masses[:, None] * inp.velocities ** 2).sum()),
                 e.get("bonds", 0.0), 0.0, e.get("angles", 0.0), 0.0, 0.0]
        return {"forces": f, "energies": np.array(terms)}
    s, x, gen = _frame_inputs(case, seed)
    top, box = _Topology(s), _t(s.box)
    theta = [_t(s.charges), _t(np.diag(s.sigma).copy()), _t(np.diag(s.epsilon).copy())]
    for p in theta:
        p.requires_grad_()
    if kind == "matching":
        ref = _reference_forces(s, x, seed)
    else:
        ge, gf = _cotangents(case, x, gen)
    rows, total = [], [torch.zeros_like(p) for p in theta]
    for k in range(case["count"]):
        xk = x[k].clone().requires_grad_()
        u = sum(top.energy(xk, box, top.pairs(x[k], box, s.cutoff), *theta).values())
        f = -torch.autograd.grad(u, xk, create_graph=True)[0]
        if kind == "matching":
            loss = ((f - ref[k]) ** 2).sum()
            grads = torch.autograd.grad(loss, theta, allow_unused=True)
            rows.append((float(loss.detach()),))
        else:
            loss = ge[k] * u + (gf[k] * f).sum()
            dx, *grads = torch.autograd.grad(loss, [xk] + theta)
            rows.append((float(u.detach()), f.detach(), dx))
        total = [t + g for t, g in zip(total, grads)]
    out = dict(zip(("charges", "sigma", "epsilon"), total))
    if kind == "matching":
        return dict(out, loss=np.array([r[0] for r in rows]))
    return dict(out, energy=np.array([r[0] for r in rows]), forces=torch.stack([r[1] for r in rows]),
                positions=torch.stack([r[2] for r in rows]))
