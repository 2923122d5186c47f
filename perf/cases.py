"""The work that a program using this framework has it do, as a list of cases.

A case is a dict of plain values; `prepare` makes the configured system (a
`mddem_amd.hip.System` with its particles uploaded), `run` is one pass of a
program's main loop: it advances the system some steps (or one force pass)
and takes the state, as a program does between two frames of a trajectory.
A system goes on from pass to pass, as it does in such a loop.

`exact` follows the first pass in 64 bits with plain torch, from the physics
alone (all pairs inside the cutoff, no neighbor lists or images of the
framework), in the framework's particle order: particles are put in bin order
when the first step has moved them and whenever one has used up the skin.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mddem_amd import hip
from mddem_amd import workloads as W


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # A granular gas of 500 spheres, the reference's own DEM benchmark size, with the
        # defaults of the API: the smallest system, bound by launches.
        dict(name="gas_500", kind="gas", n=500, phi=0.134, precision="mixed", box_exit=True,
             steps=500),
        # A middling gas in 64 bits: a serving job near the low end of its range.
        dict(name="gas_20k_fp64", kind="gas", n=19683, phi=0.2, precision="fp64",
             box_exit=False, steps=400),
        # The largest gas of the serving stream.
        dict(name="gas_200k", kind="gas", n=200000, phi=0.134, precision="mixed",
             box_exit=False, steps=400),
        # A batch of independent gases of uneven size in one context, with the launch shape
        # that the ensemble driver's tuner picks for dilute gases.
        dict(name="ensemble_64", kind="ensemble", nsys=64, nmin=200, nmax=20000,
             precision="mixed", steps=200),
        # The settled bed of the DEM headline, 4,000,000 spheres on a plane under gravity, at
        # the launch shape that the benchmark picks.
        dict(name="bed_4m", kind="bed", base=62500, tiles=8, model="plain", lanes=0,
             precision="mixed", steps=300),
        # A smaller bed in 64 bits with the API's default launch shape.
        dict(name="bed_250k_fp64", kind="bed", base=62500, tiles=2, model="plain", lanes=-1,
             precision="fp64", steps=300),
        # Cohesive spheres with rolling resistance: the optional contact models.
        dict(name="bed_140k_cohesive", kind="bed", base=35000, tiles=2, model="cohesive",
             lanes=-1, precision="fp64", steps=200),
        # A small LJ fluid under the reference's rebuild rule (a rebuild whenever an atom
        # leaves the box): nearly every step rebuilds.
        dict(name="lj_4k_box_exit", kind="lj", ncell=10, rho=0.85, temperature=0.85,
             thermostat=True, precision="fp64", box_exit=True, steps=50),
        # A thermostatted LJ fluid at the README's 32,000 atoms, lazily wrapped.
        dict(name="lj_32k", kind="lj", ncell=20, rho=0.85, temperature=0.85, thermostat=True,
             precision="mixed", box_exit=False, steps=100),
        # The LJ headline: 256,000 atoms, thermostatted, mixed precision.
        dict(name="lj_256k", kind="lj", ncell=40, rho=0.85, temperature=0.85, thermostat=True,
             precision="mixed", box_exit=False, steps=100),
        # The largest LJ size of the serving stream without a thermostat, in 64 bits.
        dict(name="lj_500k_nve_fp64", kind="lj", ncell=50, rho=0.85, temperature=0.85,
             thermostat=False, precision="fp64", box_exit=False, steps=50),
        # One call per reference system, as a host program that keeps its own step loop
        # makes them: neighbor list, pair forces, the forces on the host, an odd size.
        dict(name="lj_list_force_99k", kind="list_force", ncell=29, rho=0.85, temperature=0.85,
             precision="mixed"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["gas", "gas", "ensemble", "bed", "bed", "lj", "lj", "lj", "list_force"])
    precision = rng.choice(["mixed", "fp64"])
    if kind == "gas":
        n = int(_log_uniform(rng, 500, 200000))
        return dict(kind=kind, n=n, phi=round(rng.uniform(0.05, 0.3), 3), precision=precision,
                    box_exit=rng.random() < 0.3, steps=rng.randrange(100, 401))
    if kind == "ensemble":
        nmax = int(_log_uniform(rng, 1000, 20000))
        return dict(kind=kind, nsys=rng.randrange(16, 65), nmin=200, nmax=nmax,
                    precision=precision, steps=rng.randrange(100, 201))
    if kind == "bed":
        model = rng.choice(["plain", "plain", "cohesive"])
        return dict(kind=kind, base=rng.randrange(20001, 62501),
                    tiles=rng.randrange(1, 7 if model == "plain" else 3), model=model,
                    lanes=rng.choice([-1, 0]), precision=precision,
                    steps=rng.randrange(50, 301))
    ncell = int(round(_log_uniform(rng, 6, 50)))
    case = dict(kind=kind, ncell=ncell, rho=round(rng.uniform(0.8, 0.9), 3),
                temperature=round(rng.uniform(0.7, 1.2), 3), precision=precision)
    if kind == "lj":
        case.update(thermostat=rng.random() < 0.6, box_exit=ncell <= 12 and rng.random() < 0.4,
                    steps=rng.randrange(40, 61) if ncell > 35 else rng.randrange(50, 101))
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _bed(case, seed):
    """A deposited bed on a 0.05 m square, repeated tiles x tiles (the box is
    periodic in x and y, so the repeated bed is a bed of the larger box)."""
    side = 0.05
    w = W.dem_packed_bed(n=case["base"], box=(side, side, 1.2), seed=W.SEED_BASE + 1000 + seed)
    m = case["tiles"]
    # (moved off the lattice lines, so that no sphere sits exactly on a periodic face, where
    # the reference lists a pair once from each side)
    parts = [w.pos + np.array([ix * side + 1.7e-4, iy * side + 2.3e-4, 0.0])
             for ix in range(m) for iy in range(m)]
    w.pos = np.concatenate(parts)
    w.pos[:, :2] = np.mod(w.pos[:, :2], m * side)
    rep = m * m
    n = w.pos.shape[0]
    w.vel = np.zeros((n, 3))
    w.omega = np.zeros((n, 3))
    w.radius = np.tile(w.radius, rep)
    w.mass = np.tile(w.mass, rep)
    w.cutoff_radius = np.tile(w.cutoff_radius, rep)
    w.atype = np.zeros(n, np.uint32)
    w.hi = np.array([m * side, m * side, 1.2])
    return w


def _gas(n, phi, restitution, friction, seed):
    """A gas as it is some time after its start, with pairs about to collide:
    spheres that are each other's nearest neighbor are moved together to a
    gap below 40 micrometres (a few hundred steps of flight), where that
    brings neither of them into another sphere."""
    w = W.gas_system(n, phi, restitution, friction, seed=seed)
    x0, r, L = _t(w.pos), _t(w.radius), _t(w.hi)
    i, j = _close_pairs(x0, 2.0 * r, w.hi, w.periodic)

    def sep(x, a, b):
        d = x[b] - x[a]
        return d - L * torch.round(d / L)

    dist = sep(x0, i, j).norm(dim=1)
    near = torch.full((n,), math.inf, dtype=torch.float64, device="cuda")
    near.scatter_reduce_(0, i, dist, "amin")
    near.scatter_reduce_(0, j, dist, "amin")
    both = (dist == near[i]) & (dist == near[j])
    pi, pj, pd = i[both], j[both], dist[both]
    gap = 4e-5 * _t(W.Stream(seed + 1).uniform(n))[pi]
    shift = (0.5 * (pd - 2.0 * r[pi] - gap)).clamp(min=0.0)[:, None] * (sep(x0, pi, pj) / pd[:, None])
    move = torch.zeros_like(x0)
    move[pi] = shift
    move[pj] = -shift
    mate = torch.arange(n, device="cuda")
    mate[pi], mate[pj] = pj, pi
    for _ in range(20):
        bad = sep(x0 + move, i, j).norm(dim=1) < 2.0 * r[i]
        if not bool(bad.any()):
            break
        hit = torch.cat([i[bad], j[bad]])
        move[hit] = 0.0
        move[mate[hit]] = 0.0
    w.pos = torch.remainder(x0 + move, L).cpu().numpy()
    return w


def _workload(case, seed):
    kind = case["kind"]
    if kind == "gas":
        return _gas(case["n"], case["phi"], 0.95, 0.4, W.SEED_BASE + 2000 + 2 * seed)
    if kind == "bed":
        return _bed(case, seed)
    w = W.lj_fcc(ncell=case["ncell"], rho=case["rho"], temperature=case["temperature"],
                 seed=W.SEED_BASE + 3000 + seed, thermostat=case.get("thermostat", False))
    if kind == "list_force":  # off the lattice sites, as in a run
        st = W.Stream(W.SEED_BASE + 5000 + seed)
        w.pos = np.mod(w.pos + 0.04 * st.normal(3 * w.n).reshape(-1, 3), w.hi)
    return w


def _ensemble(case, seed):
    """Sizes, densities and materials as the ensemble workload draws them (the
    same for every seed), the spheres from the seed."""
    lo, hi = case["nmin"], case["nmax"]
    u = W.Stream(W.SEED_BASE + 4000).uniform(4 * case["nsys"]).reshape(-1, 4)
    out = []
    for k in range(case["nsys"]):
        n = int(round(lo * math.exp(u[k, 0] * math.log(hi / lo))))
        out.append(_gas(n, 0.05 + 0.25 * u[k, 3], 0.7 + 0.29 * u[k, 1], 0.1 + 0.5 * u[k, 2],
                        ((W.SEED_BASE + 4001 + seed) << 12) + 2 * k))
    return out


COHESIVE = dict(rolling_friction=0.2, rolling_stiffness=2e-2, rolling_damping=1e-8,
                cohesion_energy=5e3)


def prepare(case, seed):
    prec = hip.MIXED if case["precision"] == "mixed" else hip.FP64
    kind = case["kind"]
    if kind == "ensemble":
        systems = _ensemble(case, seed)
        w0 = systems[0]
        s = hip.System(hip.MODEL_DEM, prec)
        cut = 2.0 * float(w0.cutoff_radius[0]) * w0.skin_fraction
        s.set_neighbor(w0.skin_fraction, 1.5 * cut, 0, True, 1000, True)
        s.set_rebuild_on_box_exit(False)
        s.set_dt(w0.dt)
        s.set_force_lanes(0)
        s.set_dem_wave(False)
        for w in systems:
            m = w.materials
            s.add_system(w.lo, w.hi, m["youngs"][0], m["poisson"][0], m["restitution"][0],
                         m["friction"][0], w.pos, w.vel, w.mass, w.cutoff_radius, w.radius,
                         omega=w.omega, tag=w.tag)
        s.nsystems()  # uploads the added systems
    else:
        w = _workload(case, seed)
        s = hip.from_workload(w, prec, box_exit=case.get("box_exit", False))
        if kind == "bed":
            if case["lanes"] >= 0:
                s.set_force_lanes(case["lanes"])
            if case["model"] == "cohesive":
                s.set_material_extras(**{k: [v] for k, v in COHESIVE.items()})
                s.set_contact_models(rolling_sds=True)
    return dict(system=s, steps=case.get("steps", 0), kind=kind)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    s = state["system"]
    if state["kind"] == "list_force":
        s.bin_neighbor_list()
        s.lj_force()
        force, _ = s.forces()
        return dict(force=force)
    s.run(state["steps"])
    return s.state()


def work(case):
    """Bytes: the state that a step has to read and write once (position, velocity, force;
    spin and torque for spheres) and one word per half-list pair, each step, and the state
    taken at the end. Operations: about 30 per LJ pair inside the cutoff, 200 per contact."""
    fb = 4.0 if case["precision"] == "mixed" else 8.0
    kind = case["kind"]
    if kind in ("lj", "list_force"):
        n = 4.0 * case["ncell"] ** 3
        half = 0.5 * case["rho"] * 4.0 / 3.0 * math.pi
        k_list, k_cut = half * 2.8 ** 3, half * 2.5 ** 3
        if kind == "list_force":
            return dict(bytes=n * (24 + 3 * fb + 8 * k_list + 24), flops=n * 30 * k_cut)
        steps = case["steps"]
        # x, v read and written, 1/m, F written by the force pass and read by the kicks
        step = n * (96 + 8 + 6 * fb + 4 * k_list)
        return dict(bytes=steps * step + n * 64, flops=steps * n * 30 * k_cut)
    steps = case["steps"]
    if kind == "bed":
        n, k, c = float(case["base"] * case["tiles"] ** 2), 2.2, 1.0
    elif kind == "gas":
        n, k, c = float(case["n"]), 8.0 * case["phi"] * 0.5, 0.05
    else:
        lo, hi = case["nmin"], case["nmax"]
        n = case["nsys"] * (hi - lo) / math.log(hi / lo)
        k, c = 8.0 * 0.175 * 0.5, 0.05
    step = n * (96 + 48 + 16 + 12 * fb + 4 * k + 56 * c)
    return dict(bytes=steps * step + n * 120, flops=steps * n * (60 + 20 * k + 200 * c))


# ---------------------------------------------------------------------------
# the first pass in 64 bits
# ---------------------------------------------------------------------------

def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64), device="cuda")


def _bin_key(x, w, mn, mx):
    """Bin of each particle: the reference's bin grid (bins no smaller than the
    pair cutoff, a margin of bins around the box)."""
    cut = 2.0 * mx * w.skin_fraction
    gcut = max(cut + 2.0 * (w.skin_fraction - 1.0) * mn, cut)
    size = max(w.bin_size, cut)
    key = torch.zeros(x.shape[0], dtype=torch.int64, device=x.device)
    for d in range(3):
        L = float(w.hi[d] - w.lo[d])
        nb = int(max(math.floor(L / size), 1))
        bs = L / nb
        sl = math.ceil(gcut / bs) + math.ceil(cut / bs)
        nd = nb + 2 * sl
        c = torch.floor((x[:, d] - (float(w.lo[d]) - bs * sl)) * (1.0 / bs)).long()
        key = key * nd + c.clamp(0, nd - 1)
    return key


def _close_pairs(x, reach, L, periodic):
    """All pairs i < j (one image each, the nearest) with |d| < reach_i + reach_j."""
    dev = x.device
    n = x.shape[0]
    cut = 2.0 * float(reach.max())
    nc = [max(int(math.floor(float(L[d]) / cut)), 1) for d in range(3)]
    c = [(x[:, d] / float(L[d]) * nc[d]).floor().long() for d in range(3)]
    c = [c[d] % nc[d] if periodic[d] else c[d].clamp(0, nc[d] - 1) for d in range(3)]
    key = (c[0] * nc[1] + c[1]) * nc[2] + c[2]
    skey, order = torch.sort(key, stable=True)
    cells = torch.arange(nc[0] * nc[1] * nc[2] + 1, device=dev)
    start = torch.searchsorted(skey, cells)
    me = torch.arange(n, device=dev)
    Lt = torch.tensor([float(v) for v in L], dtype=torch.float64, device=dev)
    per = torch.tensor([1.0 if p else 0.0 for p in periodic], dtype=torch.float64, device=dev)
    offs = [[0], [0, 1]]
    axis = [offs[nc[d] - 1] if nc[d] <= 2 else [-1, 0, 1] for d in range(3)]
    out_i, out_j = [], []
    for ox in axis[0]:
        for oy in axis[1]:
            for oz in axis[2]:
                ok = torch.ones(n, dtype=torch.bool, device=dev)
                q = []
                for d, o in ((0, ox), (1, oy), (2, oz)):
                    v = c[d] + o
                    if periodic[d]:
                        v = v % nc[d]
                    else:
                        ok &= (v >= 0) & (v < nc[d])
                        v = v.clamp(0, nc[d] - 1)
                    q.append(v)
                nk = (q[0] * nc[1] + q[1]) * nc[2] + q[2]
                s0 = start[nk]
                cnt = torch.where(ok, start[nk + 1] - s0, 0)
                for m in range(int(cnt.max())):
                    i = me[cnt > m]
                    j = order[s0[i] + m]
                    keep = j > i
                    i, j = i[keep], j[keep]
                    dv = x[j] - x[i]
                    dv -= per * Lt * torch.round(dv / Lt)
                    r = reach[i] + reach[j]
                    keep = (dv * dv).sum(1) < r * r
                    out_i.append(i[keep])
                    out_j.append(j[keep])
    return torch.cat(out_i), torch.cat(out_j)


class _Order:
    """Wrapping and bin order as the step loop keeps them: at the first step
    and whenever a particle has moved half the skin since (or, with box_exit,
    has left the periodic box)."""

    def __init__(self, w, box_exit):
        self.w, self.box_exit = w, box_exit
        self.L = _t(w.hi - w.lo)
        self.lo = _t(w.lo)
        self.per = torch.tensor([bool(p) for p in w.periodic], device="cuda")
        self.mn, self.mx = float(w.cutoff_radius.min()), float(w.cutoff_radius.max())
        self.thr2 = ((w.skin_fraction - 1.0) * self.mn) ** 2
        self.built = None

    def due(self, x):
        if self.built is None:
            return True
        d = x - self.built
        d = d - torch.where(self.per, self.L * torch.round(d / self.L), 0.0)
        if bool(((d * d).sum(1) > self.thr2).any()):
            return True
        if not self.box_exit:
            return False
        return bool((self.per & ((x < self.lo) | (x >= self.lo + self.L))).any())

    def rebuild(self, x):
        """(wrapped positions in the new order, the order)"""
        x = torch.where(self.per & (x < self.lo), x + self.L,
                        torch.where(self.per & (x >= self.lo + self.L), x - self.L, x))
        order = torch.sort(_bin_key(x, self.w, self.mn, self.mx), stable=True)[1]
        self.built = x[order].clone()
        return x[order], order


def _lj_force(x, i, j, L, cut2):
    d = x[j] - x[i]
    d -= L * torch.round(d / L)
    r2 = (d * d).sum(1)
    inv = 1.0 / r2
    r6 = inv * inv * inv
    fp = torch.where(r2 < cut2, inv * r6 * (48.0 * r6 - 24.0), 0.0)
    fd = fp[:, None] * d
    f = torch.zeros_like(x)
    f.index_add_(0, i, fd, alpha=-1.0)
    f.index_add_(0, j, fd)
    return f


def _lj_exact(w, case):
    x, v = _t(w.pos), _t(w.vel)
    n, dt, L = w.n, w.dt, _t(w.hi - w.lo)
    keep = _Order(w, case.get("box_exit", False))
    if case["kind"] == "list_force":
        x, _ = keep.rebuild(x)
        i, j = _close_pairs(x, torch.full((n,), 1.25, dtype=torch.float64, device="cuda"),
                            w.hi - w.lo, (True,) * 3)
        return dict(force=_lj_force(x, i, j, L, 6.25).cpu().numpy())
    f = torch.zeros_like(x)
    nh = w.nose_hoover is not None
    if nh:
        temp, tau = w.nose_hoover
        ndof = 3.0 * n - 3.0
        q_mass = ndof * temp * tau * tau
    p_xi, scale = 0.0, 1.0
    margin = 0.5
    at = None
    for s in range(case["steps"]):
        if nh:
            term = dt / 2.0 * (float((v * v).sum()) - ndof * temp)
            p_xi += term if s == 0 else 2.0 * term
            scale = math.exp(-dt / 2.0 * p_xi / q_mass)
            v = v * scale
        v = v + (0.5 * dt) * f
        x = x + v * dt
        if keep.due(x):
            x, order = keep.rebuild(x)
            v = v[order]
            if at is not None:  # the pair list keeps up with the new order
                at = at[order]
                back = torch.empty_like(order)
                back[order] = torch.arange(n, device="cuda")
                i, j = back[i], back[j]
        if at is not None:
            d = x - at
            d -= L * torch.round(d / L)
        if at is None or float((d * d).sum(1).max()) > (0.5 * margin) ** 2:
            reach = torch.full((n,), 0.5 * (2.5 + margin), dtype=torch.float64, device="cuda")
            i, j = _close_pairs(x, reach, w.hi - w.lo, (True,) * 3)
            at = x.clone()
        f = _lj_force(x, i, j, L, 6.25)
        v = (v + (0.5 * dt) * f) * scale
    return dict(tag=None, image=None, pos=x.cpu().numpy(), vel=v.cpu().numpy())


SQRT_5_3 = 0.9128709291752768  # the reference's damping constant


def _cross(a, b):
    return torch.linalg.cross(a, b, dim=1)


def _dem_exact(w, case):
    """None if particles rebuild again within the pass (the springs' owners
    would have to be followed)."""
    x, v = _t(w.pos), _t(w.vel)
    m, r = _t(w.mass), _t(w.radius)
    n, dt = w.n, w.dt
    om = torch.zeros_like(x)
    quat = torch.zeros((n, 4), dtype=torch.float64, device="cuda")
    quat[:, 0] = 1.0
    inertia = 0.4 * m * r * r
    f, tq = torch.zeros_like(x), torch.zeros_like(x)
    per = torch.tensor([bool(p) for p in w.periodic], device="cuda")
    L = _t(w.hi - w.lo)
    e, nu = float(w.materials["restitution"][0]), float(w.materials["poisson"][0])
    young, mu = float(w.materials["youngs"][0]), float(w.materials["friction"][0])
    beta = -math.log(e) / math.sqrt(math.pi ** 2 + math.log(e) ** 2)
    e_eff = young / (2.0 * (1.0 - nu * nu))
    g_eff = young / (4.0 * (2.0 - nu) * (1.0 + nu))
    extra = COHESIVE if case.get("model") == "cohesive" else None
    keep = _Order(w, case.get("box_exit", False))
    for s in range(case["steps"]):
        v = v + (0.5 * dt) * f / m[:, None]
        x = x + v * dt
        om = om + (0.5 * dt) * tq / inertia[:, None]
        mag = om.norm(dim=1, keepdim=True)
        half = 0.5 * dt * mag
        ax = torch.where(mag * dt > 1e-14, om / mag.clamp(min=1e-300), 0.0) * torch.sin(half)
        a0 = torch.where(mag * dt > 1e-14, torch.cos(half), 1.0)
        b0, bv = quat[:, :1].clone(), quat[:, 1:].clone()
        quat = torch.cat([a0 * b0 - (ax * bv).sum(1, keepdim=True),
                          a0 * bv + ax * b0 + _cross(ax, bv)], dim=1)
        if keep.due(x):
            if s > 0:
                return None
            x, o = keep.rebuild(x)
            v, om, quat, m, r, inertia = v[o], om[o], quat[o], m[o], r[o], inertia[o]
            ci, cj = _close_pairs(x, r * w.skin_fraction, w.hi - w.lo, w.periodic)
            tag = o
            swap = tag[ci] > tag[cj]  # springs live in the lower tag's frame
            ci, cj = torch.where(swap, cj, ci), torch.where(swap, ci, cj)
            spring = torch.zeros((ci.shape[0], 3), dtype=torch.float64, device="cuda")
            roll = torch.zeros_like(spring)
        f, tq = torch.zeros_like(x), torch.zeros_like(x)
        d = x[cj] - x[ci]
        d = d - torch.where(per, L * torch.round(d / L), 0.0)
        dist2 = (d * d).sum(1)
        sum_r = r[ci] + r[cj]
        hit = dist2 < sum_r * sum_r
        spring[~hit] = 0.0
        roll[~hit] = 0.0
        k = torch.nonzero(hit).flatten()
        if k.numel():
            i, j, d = ci[k], cj[k], d[k]
            dist = dist2[k].sqrt()[:, None]
            nrm = d / dist
            ri, rj = r[i][:, None], r[j][:, None]
            delta = torch.minimum(ri + rj - dist, 0.5 * torch.minimum(ri, rj))
            r_eff = ri * rj / (ri + rj)
            m_r = 1.0 / (1.0 / m[i] + 1.0 / m[j])[:, None]
            sdr = torch.sqrt(delta * r_eff)
            s_n, k_n, k_t = 2.0 * e_eff * sdr, 4.0 / 3.0 * e_eff * sdr, 8.0 * g_eff * sdr
            vr = (v[j] - _cross(om[j], rj * nrm)) - (v[i] + _cross(om[i], ri * nrm))
            v_n = (vr * nrm).sum(1, keepdim=True)
            fn = k_n * delta - 2.0 * beta * SQRT_5_3 * torch.sqrt(s_n * m_r) * v_n
            if extra:
                fn = fn - extra["cohesion_energy"] * math.pi * delta * r_eff
            else:
                fn = fn.clamp(min=0.0)
            vt = vr - v_n * nrm
            sp = spring[k]
            sp = sp - (sp * nrm).sum(1, keepdim=True) * nrm + vt * dt
            lim = mu * fn.abs()
            mag = k_t * sp.norm(dim=1, keepdim=True)
            sp = torch.where((mag > lim) & (mag > 1e-30), sp * (lim / mag.clamp(min=1e-300)), sp)
            ft = k_t * sp - 2.0 * SQRT_5_3 * beta * torch.sqrt(k_t * m_r) * vt
            mag = ft.norm(dim=1, keepdim=True)
            ft = torch.where((mag > lim) & (mag > 1e-30), ft * (lim / mag.clamp(min=1e-300)), ft)
            spring[k] = sp
            fi = -fn * nrm + ft
            f.index_add_(0, i, fi)
            f.index_add_(0, j, fi, alpha=-1.0)
            t = _cross(nrm, ft)
            ti, tj = ri * t, rj * t
            if extra:
                rel = om[i] - om[j]
                rl = rel - (rel * nrm).sum(1, keepdim=True) * nrm
                rd = roll[k]
                rd = rd - (rd * nrm).sum(1, keepdim=True) * nrm + rl * dt
                kr, gr = extra["rolling_stiffness"], extra["rolling_damping"]
                tr = -kr * rd - gr * rl
                lim = extra["rolling_friction"] * fn.abs() * r_eff
                mag = tr.norm(dim=1, keepdim=True)
                over = (mag > lim) & (mag > 1e-30)
                tr = torch.where(over, tr * (lim / mag.clamp(min=1e-300)), tr)
                roll[k] = torch.where(over, (tr + gr * rl) / -kr, rd)
                ti, tj = ti + tr, tj - tr
            tq.index_add_(0, i, ti)
            tq.index_add_(0, j, tj)
        for point, normal, _ in w.walls:
            nv = _t(normal)
            dist = ((x - _t(point)) * nv).sum(1)
            delta = torch.minimum(r - dist, 0.5 * r)
            on = (delta > 0.0) & (dist > 0.0)
            dl = delta.clamp(min=0.0)
            sdr = torch.sqrt(dl * r)
            fw = (4.0 / 3.0 * e_eff * sdr * dl - 2.0 * beta * SQRT_5_3
                  * torch.sqrt(2.0 * e_eff * sdr * m) * (v * nv).sum(1))
            if extra:
                fw = fw - extra["cohesion_energy"] * math.pi * dl * r
            else:
                fw = fw.clamp(min=0.0)
            f += torch.where(on, fw, 0.0)[:, None] * nv
        if w.gravity is not None:
            f += m[:, None] * _t(np.array(w.gravity))
        v = v + (0.5 * dt) * f / m[:, None]
        om = om + (0.5 * dt) * tq / inertia[:, None]
    host = [a.cpu().numpy() for a in (x, v, om, quat)]
    return dict(tag=None, image=None, pos=host[0], vel=host[1], omega=host[2], quat=host[3])


def exact(case, seed):
    if case["kind"] == "ensemble":
        parts = []
        for w in _ensemble(case, seed):
            w.bin_size = 1.5 * 2.0 * float(w.cutoff_radius[0]) * w.skin_fraction
            parts.append(_dem_exact(w, case))
        if any(p is None for p in parts):
            return None
        return {k: None if parts[0][k] is None else np.concatenate([p[k] for p in parts])
                for k in parts[0]}
    w = _workload(case, seed)
    return _dem_exact(w, case) if w.model == "dem" else _lj_exact(w, case)
