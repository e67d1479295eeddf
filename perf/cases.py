"""The work that a user of this framework has it do, as timed cases.

A pass is one run of a simulation through the public classes: the initial
state goes up, a number of steps run on the device, the final state comes
back (what run_system does, the initial state kept so that every pass starts
from it), or one training run of the learned propagator's network.

  gas      newton_step! of LJ gases (cut at 2.5 sigma, or the reference's
           LenJonesCfg without a cutoff) and harmonic discs, periodic or
           walled boxes
  rings    Rings step! of active-ring mixtures with device rotational noise
  active   Szabo and run-and-tumble particles with device noise
  batch    many systems of uneven size stepped together
  train    Adam steps of the network on a data set of feature rows
  learned  gated learned steps of a ring mixture (features, network, gate)

exact() restates the same physics in FP64 torch: pair sums over the 3x3
chunk block, both force evaluations of a Verlet step with the step's chunks,
the ring, self-propelled and network formulas, and the Philox streams.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "mavi.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DT = 1e-3
N_IN, N_HID, N_OUT = 160, 128, 2
LAYERS = ((N_HID, N_IN), (N_HID, N_HID), (N_HID, N_HID), (N_OUT, N_HID))
K_PLAIN, R_FEAT, S_T = 10, 1.25, 1e-3  # learned steps: plain steps each, feature radius, output unit
PHI = 0.8  # ring packing fraction


def listed():
    return [
        # one newton_step! with the state handed over and back, the
        # reference's own step loop: latency and launches
        dict(name="gas_1k_one_step", family="gas", potential="lj", walls="periodic", nx=32, ny=32, steps=1),
        # the size of the reference's examples, run between two looks at it
        dict(name="gas_1k", family="gas", potential="lj", walls="periodic", nx=32, ny=32, steps=500),
        # an ordinary system of ragged size
        dict(name="gas_100k", family="gas", potential="lj", walls="periodic", nx=331, ny=307, steps=400),
        # the framework's headline system
        dict(name="gas_1m", family="gas", potential="lj", walls="periodic", nx=1024, ny=1024, steps=400),
        # the reference's LenJonesCfg as it is: every pair in adjacent chunks
        dict(name="gas_ref_200k", family="gas", potential="lj_ref", walls="periodic", nx=451, ny=449, steps=150),
        # harmonic discs between hard walls
        dict(name="discs_walled_22k", family="gas", potential="harm", walls="rigid", nx=151, ny=149, steps=300),
        # rings: an example's size and the mixture of the framework's ring benchmark
        dict(name="rings_2k", family="rings", ring_cols=10, ring_rows=10, per_ring=20, short=0, steps=300),
        dict(name="rings_800k", family="rings", ring_cols=200, ring_rows=200, per_ring=20, short=0, steps=200),
        # self-propelled particles
        dict(name="szabo_30k", family="active", model="szabo", nx=181, ny=167, steps=200),
        # an ensemble of uneven systems, half gases and half rings
        dict(name="batch_48", family="batch", replicas=48, nmin=1000, nmax=40000, steps=200),
        # training and use of the learned propagator
        dict(name="train_8192", family="train", rows=100000, batch=8192, steps=40),
        dict(name="learned_100k", family="learned", ring_cols=72, ring_rows=70, per_ring=20, steps=40),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["gas"] * 4 + ["rings"] * 3 + ["active"] * 2 + ["batch", "train", "learned"])
    if family == "gas":
        nx = _log(rng, 9, 900)
        ny = max(9, min(1000, int(nx * rng.uniform(0.6, 1.4))))
        potential = rng.choice(["lj", "lj", "lj_ref", "harm"])
        return dict(family=family, potential=potential, walls=rng.choice(["periodic", "periodic", "rigid"]), nx=nx,
                    ny=ny, steps=rng.choice([1, 20, 50, 150, 300] if nx * ny < 20000 else [50, 150, 250]))
    if family == "rings":
        c = _log(rng, 4, 180)
        return dict(family=family, ring_cols=c, ring_rows=max(4, min(180, int(c * rng.uniform(0.6, 1.4)))),
                    per_ring=rng.randint(8, 24), short=rng.choice([0, 0, 2, 5]), steps=rng.choice([20, 60, 150]))
    if family == "active":
        nx = _log(rng, 16, 200)
        return dict(family=family, model=rng.choice(["szabo", "rtp"]), nx=nx,
                    ny=max(16, min(180, int(nx * rng.uniform(0.6, 1.4)))), steps=rng.choice([20, 60, 150]))
    if family == "batch":
        return dict(family=family, replicas=rng.randint(4, 40), nmin=1000, nmax=rng.randint(4000, 32000),
                    steps=rng.choice([50, 100, 150]))
    if family == "train":
        return dict(family=family, rows=_log(rng, 2000, 100000), batch=_log(rng, 256, 12000), steps=rng.randint(10, 40))
    c = _log(rng, 8, 70)
    return dict(family=family, ring_cols=c, ring_rows=max(8, min(70, int(c * rng.uniform(0.6, 1.4)))),
                per_ring=rng.randint(12, 24), steps=rng.randint(8, 30))


# ---------------------------------------------------------------------------
# Inputs (numpy, from the seed alone)
# ---------------------------------------------------------------------------
POT = {"lj": dict(density=0.7, side=2.5), "lj_ref": dict(density=0.7, side=2.5), "harm": dict(density=0.6, side=1.25)}
HARM = dict(k_rep=10.0, k_atr=1.0, dist_eq=1.0, dist_max=1.2)
SZABO = dict(vo=1.0, mobility=1.0, relax_time=1.0, k_rep=10.0, k_adh=0.75, r_eq=1.0, r_max=1.1, rot_diff=0.01)
RTP = dict(vo=1.0, sigma=1.0, epsilon=1.0, tumble_rate=1.0)
RING = dict(relax_time=1.0, vo=1.0, mobility=1.0, rot_diff=0.1, k_area=1.0, k_spring=20.0, l_spring=1.0)
RING_PAIR = dict(k_rep=10.0, k_atr=0.0, dist_eq=1.0, dist_max=1.0)


def _lattice(rng, nx, ny, a, jitter):
    ix, iy = np.meshgrid(np.arange(nx), np.arange(ny), indexing="xy")
    pos = np.stack([(ix.ravel() + 0.5) * a, (iy.ravel() + 0.5) * a], axis=1)
    pos += rng.uniform(-jitter, jitter, size=pos.shape)
    return pos, nx * a, ny * a


def _gas_inputs(case, seed):
    """A jittered lattice with Gaussian velocities of temperature 1."""
    rng = np.random.default_rng(seed)
    p = POT[case["potential"]]
    pos, L, H = _lattice(rng, case["nx"], case["ny"], p["density"] ** -0.5, 0.1 if case["walls"] == "periodic" else 0.03)
    vel = rng.standard_normal(pos.shape)
    vel -= vel.mean(axis=0)
    return dict(pos=pos, vel=vel, L=L, H=H, cols=int(L // p["side"]), rows=int(H // p["side"]))


def _ring_inputs(case, seed, chunk=1.0):
    """Two types of rings (the second up to `short` particles smaller, its
    target area contracted to 0.9) on a lattice at packing fraction PHI, the
    centres, angles and particles jittered so that neighbouring rings touch."""
    rng = np.random.default_rng(seed)
    cols, rows, nper = case["ring_cols"], case["ring_rows"], case["per_ring"]
    nr = cols * rows
    types = rng.integers(1, 3, size=nr).astype(np.int32)
    counts = np.array([nper, max(4, nper - case.get("short", 0))])
    radius = 1.0 / (2 * math.sin(math.pi / nper))
    spacing = math.sqrt(math.pi / PHI) * (radius + 0.5)
    L, H = cols * spacing, rows * spacing
    k = np.arange(nr)
    centres = np.stack([(k % cols + 0.5) * spacing, (k // cols + 0.5) * spacing], axis=1)
    centres += rng.uniform(-0.12, 0.12, size=centres.shape)
    n_of = counts[types - 1]
    r_of = 0.97 / (2 * np.sin(math.pi / n_of))
    ang = (np.arange(nper)[None, :] / n_of[:, None] + rng.random(nr)[:, None]) * 2 * math.pi
    pos = centres[:, None, :] + r_of[:, None, None] * np.stack([np.cos(ang), np.sin(ang)], axis=2)
    pos += rng.uniform(-0.02, 0.02, size=pos.shape)
    pos = np.mod(pos, np.array([L, H]))
    pol = rng.random(nr) * 2 * math.pi
    area = counts / (4 * np.tan(math.pi / counts))
    p0 = counts / np.sqrt(area * np.array([1.0, 0.9]))
    return dict(pos=pos, pol=pol, types=types, counts=counts, p0=p0, L=L, H=H, cols=int(L // chunk),
                rows=int(H // chunk))


def _active_inputs(case, seed):
    rng = np.random.default_rng(seed)
    if case["model"] == "szabo":
        a, jitter, side = SZABO["r_eq"], 0.05, SZABO["r_max"]
    else:
        a, jitter, side = 0.8 ** -0.5, 0.02, 2 ** (1 / 6) * RTP["sigma"]
    pos, L, H = _lattice(rng, case["nx"], case["ny"], a, jitter)
    ang = rng.random(len(pos)) * 2 * math.pi
    return dict(pos=pos, ang=ang, L=L, H=H, cols=int(L // side), rows=int(H // side))


def _batch_inputs(case, seed):
    """Replica sizes log-uniform in [nmin, nmax] (the same for every seed): LJ gases and ring mixtures in turn."""
    rng = np.random.default_rng(case["replicas"])
    out = []
    for i in range(case["replicas"]):
        n = math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"])))
        if i % 2 == 0:
            nx = max(9, int(round(math.sqrt(n))))
            sub = dict(potential="lj", walls="periodic", nx=nx, ny=max(9, int(n / nx)))
            out.append(("gas", _gas_inputs(sub, seed + 1 + i)))
        else:
            c = max(4, int(round(math.sqrt(n / 20))))
            sub = dict(ring_cols=c, ring_rows=max(4, int(n / 20 / c)), per_ring=20)
            out.append(("rings", _ring_inputs(sub, seed + 1 + i)))
    return out


def _net_params(seed):
    rng = np.random.default_rng(seed)
    out = []
    for nout, nin in LAYERS:
        a = math.sqrt(6.0 / (nin + nout))
        out += [rng.uniform(-a, a, size=nout * nin), rng.uniform(-0.05, 0.05, size=nout)]
    return np.concatenate(out).astype(np.float32)


def _train_inputs(case, seed):
    """Feature rows as the propagator makes them (14 self features, a few
    neighbour groups of 4, zeros past them) and a smooth target with noise."""
    rng = np.random.default_rng(seed)
    n = case["rows"]
    x = np.zeros((n, N_IN), dtype=np.float32)
    x[:, :14] = rng.normal(scale=0.6, size=(n, 14))
    nb = rng.poisson(3, size=n).clip(0, 12)
    g = rng.normal(scale=0.7, size=(n, 12, 4)).astype(np.float32)
    g *= (np.arange(12)[None, :] < nb[:, None])[:, :, None]
    x[:, 32:80] = g.reshape(n, 48)
    t = np.stack([np.sin(x[:, 2]) + 0.3 * x[:, 6] * x[:, 7], np.cos(x[:, 3]) - 0.5 * x[:, 32]], axis=1)
    t += rng.normal(scale=0.1, size=t.shape)
    bits = torch.from_numpy(x).to(torch.bfloat16)
    return bits.view(torch.int16).numpy().view(np.uint16), bits.to(torch.float64).numpy(), t.astype(np.float32)


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def _box(mv, d, walls="periodic"):
    wall = mv.PeriodicWalls() if walls == "periodic" else mv.RigidWalls()
    return mv.SpaceCfg(wall_type=wall, geometry_cfg=mv.RectangleCfg(length=d["L"], height=d["H"]))


def _int_cfg(mv, d):
    return mv.IntCfg(dt=DT, chunks_cfg=mv.ChunksCfg(num_cols=d["cols"], num_rows=d["rows"]), device=mv.GPU())


def _gas_dyn(mv, potential):
    if potential == "harm":
        return mv.HarmTruncCfg(**HARM)
    return mv.LenJonesCfg(sigma=1.0, epsilon=1.0, cutoff=2.5 if potential == "lj" else None)


def _ring_state(d):
    from mavi_hip import rings

    return rings.RingsState(rings_pos=d["pos"].copy(), pol=d["pol"], num_particles=[int(c) for c in d["counts"]],
                            types=d["types"])


def _ring_cfg(d):
    from mavi_hip import rings

    two = {k: [v, v] for k, v in RING.items()}
    return rings.RingsCfg(p0=[float(p) for p in d["p0"]], interaction_finder=rings.HarmTruncCfg(**RING_PAIR),
                          num_particles=[int(c) for c in d["counts"]], **two)


def prepare(case, seed):
    import mavi_hip as mv
    from mavi_hip import batch, learned, rings

    family = case["family"]
    if family == "gas":
        d = _gas_inputs(case, seed)
        first, last = (mv.SecondLawState(pos=d["pos"], vel=d["vel"]) for _ in range(2))
        system = mv.System(state=first, space_cfg=_box(mv, d, case["walls"]),
                           dynamic_cfg=_gas_dyn(mv, case["potential"]), int_cfg=_int_cfg(mv, d))
        return dict(case=case, system=system, first=first, last=last)
    if family == "active":
        d = _active_inputs(case, seed)
        dyn = mv.SzaboCfg(**SZABO) if case["model"] == "szabo" else mv.RunTumbleCfg(**RTP)
        first, last = (mv.SelfPropelledState(pos=d["pos"], pol_angle=d["ang"]) for _ in range(2))
        system = mv.System(state=first, space_cfg=_box(mv, d), dynamic_cfg=dyn, int_cfg=_int_cfg(mv, d), seed=seed)
        return dict(case=case, system=system, first=first, last=last)
    if family in ("rings", "learned"):
        d = _ring_inputs(case, seed, 1.0 if family == "rings" else R_FEAT)
        first, last = _ring_state(d), _ring_state(d)
        system = rings.RingsSystem(state=first, space_cfg=_box(mv, d), dynamic_cfg=_ring_cfg(d),
                                   int_cfg=_int_cfg(mv, d), seed=seed)
        st = dict(case=case, system=system, first=first, last=last)
        if family == "learned":
            net = learned.MLP(ctx=system.ctx)
            net.params = _net_params(seed)
            st["step"] = learned.Learned(system.dev, net, k=K_PLAIN, r_feat=R_FEAT, target_scale=S_T, seed=seed)
        return st
    if family == "batch":
        b, states = batch.Batch(), []
        for i, (kind, d) in enumerate(_batch_inputs(case, seed)):
            if kind == "gas":
                s = mv.SecondLawState(pos=d["pos"], vel=d["vel"])
                b.add(s, _box(mv, d), _gas_dyn(mv, "lj"), _int_cfg(mv, d))
                states.append((s.pos, s.vel, None))
            else:
                s = _ring_state(d)
                b.add(s, _box(mv, d), _ring_cfg(d), _int_cfg(mv, d), seed=seed + i)
                states.append((s.pos, None, s.pol))
        b.finalize()
        return dict(case=case, batch=b, states=states)
    bits, _, t = _train_inputs(case, seed)
    net = learned.MLP()
    net.params = _net_params(seed)
    net.dataset_append(bits, t)
    return dict(case=case, net=net, seed=seed)


def run(state):
    case = state["case"]
    family, steps = case["family"], case["steps"]
    if family == "train":
        net = state["net"]
        losses = net.train(steps=steps, batch=case["batch"], lr=1e-3, seed=state["seed"])
        return dict(losses=losses, params=net.params)
    if family == "batch":
        b = state["batch"]
        for i, (pos, vel, pol) in enumerate(state["states"]):
            b.upload(i, pos, vel, pol)
        b.run(steps)
        got = [b.download(i) for i in range(len(state["states"]))]
        return dict(pos=np.concatenate([p for p, _, _ in got]),
                    vel=np.concatenate([v for _, v, _ in got if v is not None]),
                    pol=np.concatenate([a for _, _, a in got if a is not None]))
    system, last = state["system"], state["last"]
    system.state = state["first"]
    system.upload()
    if family == "learned":
        state["step"].run(steps)
    else:
        system.advance(steps)
    system.state = last
    system.download()
    out = dict(pos=last.pos, forces=system.forces)
    if family == "gas":
        out["vel"] = last.vel
    elif family == "active":
        out["pol"] = last.pol_angle
    else:
        out["pol"], out["areas"] = last.pol, system.areas
        if family == "learned":  # the forces and areas belong to the last feature pass, inside the step
            out = dict(pos=last.pos, pol=last.pol)
    return out


# ---------------------------------------------------------------------------
# Work and tolerances
# ---------------------------------------------------------------------------
def _pair_flops(density, reach):
    """One evaluation, each pair once: distance, force law, two updates."""
    return 0.5 * density * math.pi * reach * reach * 24


def work(case):
    """Per step: the state read once and written once (positions, velocities
    or angles, forces), one force evaluation with each pair in range visited
    once.  Learned steps: the network's products and the plain parts.
    Training: the rows read once per step, forward and backward products."""
    family = case["family"]
    if family == "train":
        macs = sum(a * b for a, b in LAYERS)
        rows = case["batch"] * case["steps"]
        return dict(bytes=rows * (N_IN * 2 + N_OUT * 4) + case["steps"] * 24 * macs,
                    flops=rows * (6 * macs - 2 * LAYERS[0][0] * LAYERS[0][1]))
    if family == "gas":
        n = case["nx"] * case["ny"]
        reach = {"lj": 2.5, "lj_ref": 2.5, "harm": 1.2}[case["potential"]]
        return dict(bytes=case["steps"] * n * 96, flops=case["steps"] * n * (14 + _pair_flops(POT[case["potential"]]["density"], reach)))
    if family == "active":
        n = case["nx"] * case["ny"]
        return dict(bytes=case["steps"] * n * 64, flops=case["steps"] * n * (60 + _pair_flops(0.9, 1.1)))
    if family == "batch":
        # the mean of a log-uniform size
        n = case["replicas"] * (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
        return dict(bytes=case["steps"] * n * 80, flops=case["steps"] * n * (40 + _pair_flops(0.7, 2.5)))
    n = case["ring_cols"] * case["ring_rows"] * case["per_ring"]
    if family == "rings":
        return dict(bytes=case["steps"] * n * 48, flops=case["steps"] * n * (80 + _pair_flops(0.4, 1.0)))
    macs = sum(a * b for a, b in LAYERS)
    return dict(bytes=case["steps"] * n * (48 + 2 * N_IN), flops=case["steps"] * n * (2 * macs + 200))


def tolerance(case):
    """Trajectories in FP64: rounding of other summation orders grows with the
    dynamics' own instability over the steps; about four times what a change
    of order shows.  BF16 networks: rounding of activations and gradients."""
    family = case["family"]
    if family == "train":
        return {"rel": 2e-2, "max": 0.9}
    if family == "learned":
        return {"rel": 1e-6, "max": 1e-4}
    if family in ("rings", "batch"):  # the shoelace sums of far-off rings cancel
        return {"rel": 4e-9, "max": 1e-6}
    return {"rel": 1e-9, "max": 1e-6}


# ---------------------------------------------------------------------------
# The same physics in FP64 torch
# ---------------------------------------------------------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64


def _t(a, dtype=F64):
    return torch.as_tensor(np.asarray(a)).to(_DEV, dtype)


class _Space:
    """Boxes and chunk grids, one entry per particle (several systems can lie
    side by side: their chunks are numbered one after another)."""

    def __init__(self, parts, periodic=True):
        sizes = [p["n"] for p in parts]
        rep = lambda key, dt=F64: torch.cat([torch.full((n,), p[key], dtype=dt, device=_DEV) for p, n in zip(parts, sizes)])  # noqa: E731
        base = 0
        for p in parts:
            p["base"] = base
            base += p["cols"] * p["rows"]
            p["cl"], p["ch"] = p["L"] / p["cols"], p["H"] / p["rows"]
        self.L, self.H, self.cl, self.ch = rep("L"), rep("H"), rep("cl"), rep("ch")
        self.cols, self.rows, self.base = (rep(k, torch.int64) for k in ("cols", "rows", "base"))
        self.ncell, self.periodic, self.n = base, periodic, sum(sizes)

    def bins(self, pos):
        row = torch.floor((self.H - pos[:, 1]) / self.ch).to(torch.int64)
        col = torch.floor(pos[:, 0] / self.cl).to(torch.int64)
        row = torch.minimum(row, self.rows - 1).clamp(min=0)
        col = torch.minimum(col, self.cols - 1).clamp(min=0)
        cell = self.base + row * self.cols + col
        order = torch.argsort(cell, stable=True)
        count = torch.bincount(cell, minlength=self.ncell)
        return row, col, order, count, torch.cumsum(count, 0) - count, int(count.max())

    def blocks(self, bins):
        """Candidate columns of the 3x3 block: (j [n, k], valid [n, k]) per neighbour chunk."""
        row, col, order, count, start, k = bins
        q = torch.arange(k, device=_DEV)[None, :]
        me = torch.arange(self.n, device=_DEV)[:, None]
        for dr in (-1, 0, 1):
            for dc in (-1, 0, 1):
                r, c = row + dr, col + dc
                inside = torch.ones_like(r, dtype=torch.bool)
                if self.periodic:
                    r, c = torch.remainder(r, self.rows), torch.remainder(c, self.cols)
                else:
                    inside = (r >= 0) & (r < self.rows) & (c >= 0) & (c < self.cols)
                    r, c = torch.where(inside, r, row), torch.where(inside, c, col)
                cell = self.base + r * self.cols + c
                j = order[(start[cell][:, None] + q).clamp(max=self.n - 1)]
                yield j, (q < count[cell][:, None]) & inside[:, None] & (j != me)

    def image(self, dx, dy):
        if not self.periodic:
            return dx, dy
        L, H = (v if dx.dim() == 1 else v[:, None] for v in (self.L, self.H))
        return dx - L * torch.sign(dx) * (dx.abs() > L / 2), dy - H * torch.sign(dy) * (dy.abs() > H / 2)

    def wrap(self, pos):
        x, y = pos[:, 0] - self.L / 2, pos[:, 1] - self.H / 2
        return torch.stack([pos[:, 0] - self.L * torch.sign(x) * (x.abs() > self.L / 2),
                            pos[:, 1] - self.H * torch.sign(y) * (y.abs() > self.H / 2)], dim=1)

    def pair_forces(self, pos, bins, law):
        """sum_j law(r^2, j) * dr over the valid candidates."""
        f = torch.zeros_like(pos)
        for j, ok in self.blocks(bins):
            dx, dy = self.image(pos[:, 0, None] - pos[j, 0], pos[:, 1, None] - pos[j, 1])
            r2 = torch.where(ok, dx * dx + dy * dy, 1e30)
            q = law(r2, j) * ok
            f[:, 0] += (q * dx).sum(1)
            f[:, 1] += (q * dy).sum(1)
        return f


def _lj(cut):
    def law(r2, j):
        inv3 = r2 ** -3
        return torch.where(r2 <= cut * cut, (48.0 * inv3 * inv3 - 24.0 * inv3) / r2, 0.0)
    return law


def _harm(p):
    def law(r2, j):
        d = torch.sqrt(r2)
        mod = torch.where(d < p["dist_eq"], -p["k_rep"] * (d / p["dist_eq"] - 1.0), -p["k_atr"] * (d / p["dist_eq"] - 1.0))
        return torch.where(d <= p["dist_max"], mod / d, 0.0)
    return law


def _verlet_step(space, pos, vel, law, radius):
    bins = space.bins(pos)
    f1 = space.pair_forces(pos, bins, law)
    pos = pos + (vel * DT + f1 * (DT * DT / 2))
    f2 = space.pair_forces(pos, bins, law)
    vel = vel + DT / 2 * (f1 + f2)
    if space.periodic:
        return space.wrap(pos), vel, f2
    size = torch.stack([space.L, space.H], dim=1)
    return pos, torch.where((pos + radius > size) | (pos - radius < 0), -vel, vel), f2


def _mul32(a, b):
    p = a * b  # both below 2^32: the wrapped 64-bit product
    return (p >> 32) & 0xFFFFFFFF, p & 0xFFFFFFFF


def _philox(seed, step, ids, word):
    """Philox4x32-10 of (step, id, word) keyed by seed: four 32-bit words."""
    c = [torch.full_like(ids, step & 0xFFFFFFFF), torch.full_like(ids, step >> 32), ids, torch.full_like(ids, word)]
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        h0, l0 = _mul32(c[0], 0xD2511F53)
        h1, l1 = _mul32(c[2], 0xCD9E8D57)
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _normal(seed, step, ids):
    c = _philox(seed, step, ids, 0x6D617669)
    u1 = (((c[0] << 21) ^ (c[1] >> 11)).to(F64) + 1.0) * 2.0 ** -53
    u2 = (((c[2] << 21) ^ (c[3] >> 11)) & ((1 << 53) - 1)).to(F64) * 2.0 ** -53
    return torch.sqrt(-2.0 * torch.log(u1)) * torch.cos(2 * math.pi * u2)


def _uniforms(seed, step, ids):
    c = _philox(seed, step, ids, 0x72746D62)
    return [(((a << 21) ^ (b >> 11)) & ((1 << 53) - 1)).to(F64) * 2.0 ** -53 for a, b in ((c[0], c[1]), (c[2], c[3]))]


def _active_exact(case, seed):
    d = _active_inputs(case, seed)
    n = len(d["pos"])
    space = _Space([dict(d, n=n)])
    pos, th, ids = _t(d["pos"]), _t(d["ang"]), torch.arange(n, device=_DEV)
    s = SZABO

    def law(r2, j):
        dist = torch.sqrt(r2)
        mod = torch.where(dist > s["r_eq"], s["k_adh"] / s["r_eq"], s["k_rep"] / (s["r_max"] - s["r_eq"]))
        return torch.where(dist <= s["r_max"], -mod * (dist - s["r_eq"]), 0.0)

    if case["model"] == "rtp":
        law = _lj(2 ** (1 / 6))
    for step in range(1, case["steps"] + 1):
        f = space.pair_forces(pos, space.bins(pos), law)
        cs, sn = torch.cos(th), torch.sin(th)
        vx, vy = cs + f[:, 0], sn + f[:, 1]  # vo = mobility = 1
        if case["model"] == "szabo":
            cr = ((cs * vy - sn * vx) / torch.sqrt(vx.abs() + vy.abs())).clamp(-1.0, 1.0)
            th = th + torch.asin(cr) / s["relax_time"] * DT + math.sqrt(2 * s["rot_diff"] * DT) * _normal(seed, step, ids)
        else:
            u, w = _uniforms(seed, step, ids)
            th = torch.where(u < RTP["tumble_rate"] * DT, 2 * math.pi * w, th)
        pos = space.wrap(pos + torch.stack([vx, vy], dim=1) * DT)
    return dict(pos=pos, forces=f, pol=th)


class _Rings:
    """Ring mixtures side by side; all arrays over the active particles."""

    def __init__(self, parts, seeds):
        self.space = _Space([dict(p, n=int(p["counts"][p["types"] - 1].sum())) for p in parts])
        ring, prev, nxt, idx, mask, count, area0, noise = [], [], [], [], [], [], [], []
        first, r0 = 0, 0
        self.seeds, self.local, self.full = [], [], []
        for p, sd in zip(parts, seeds):
            n_of = p["counts"][p["types"] - 1].astype(np.int64)
            nmax = p["pos"].shape[1]
            start = first + np.cumsum(n_of) - n_of
            i = np.arange(nmax)[None, :]
            ok = i < n_of[:, None]
            me = start[:, None] + i
            ring.append(np.broadcast_to(r0 + np.arange(len(n_of))[:, None], ok.shape)[ok])
            prev.append(np.where(i == 0, start[:, None] + n_of[:, None] - 1, me - 1)[ok])
            nxt.append(np.where(i == n_of[:, None] - 1, start[:, None], me + 1)[ok])
            idx.append(np.broadcast_to(i, ok.shape)[ok])
            mask.append(ok)
            count.append(n_of)
            area0.append((n_of * RING["l_spring"] / p["p0"][p["types"] - 1]) ** 2)
            first += int(n_of.sum())
            r0 += len(n_of)
            self.seeds.append(sd)
            self.local.append(len(n_of))
        self.ring, self.prev, self.next, self.idx = (_t(np.concatenate(v), torch.int64) for v in (ring, prev, nxt, idx))
        self.np, self.area0 = _t(np.concatenate(count)), _t(np.concatenate(area0))
        self.mask, self.nr = mask, r0
        self.type = _t(np.concatenate([p["types"] - 1 for p in parts]), torch.int64)
        self.pos = _t(np.concatenate([p["pos"][m] for p, m in zip(parts, mask)]))
        self.pol = _t(np.concatenate([p["pol"] for p in parts]))

    def law(self, r2, j):
        p = RING_PAIR
        d = torch.sqrt(r2)
        same = self.ring[j] == self.ring[:, None]
        diff = (self.idx[j] - self.idx[:, None]).abs()
        bonded = same & ((diff == 1) | (diff == self.np[self.ring][:, None] - 1))
        return torch.where((d <= p["dist_max"]) & ~bonded, -p["k_rep"] * (d / p["dist_eq"] - 1.0) / d, 0.0)

    def diff(self, a, b):
        return torch.stack(self.space.image(a[:, 0] - b[:, 0], a[:, 1] - b[:, 1]), dim=1)

    def ring_sum(self, v):
        return torch.zeros(self.nr, dtype=F64, device=_DEV).index_add_(0, self.ring, v)

    def forces(self, bins=None):
        pos = self.pos
        f = self.space.pair_forces(pos, bins or self.space.bins(pos), self.law)
        to_next = self.diff(pos, pos[self.next])
        dist = torch.sqrt((to_next ** 2).sum(1))
        spring = (-RING["k_spring"] * (dist - RING["l_spring"]) / dist)[:, None] * to_next
        # area: shoelace over the ring's points relative to its first particle
        first = self.first()
        rel = self.unwrap(first)
        cross = rel[:, 0] * rel[self.next, 1] - rel[:, 1] * rel[self.next, 0]
        self.areas = self.ring_sum(cross) / 2
        fa = RING["k_area"] * (self.areas - self.area0)[self.ring]
        da = self.diff(pos[self.next], pos[self.prev])
        self.da = da
        f = f + spring - spring[self.prev] - fa[:, None] * torch.stack([da[:, 1], -da[:, 0]], dim=1) / 2
        return f

    def first(self):
        me = torch.arange(len(self.idx), device=_DEV)
        return (me - self.idx)

    def unwrap(self, first):
        """Points relative to the ring's first particle: running sums of the
        minimum-image steps (rings of up to 24 particles)."""
        step = self.diff(self.pos, self.pos[self.prev])
        step[self.idx == 0] = 0.0
        total = torch.cumsum(step, 0)
        return total - total[first]

    def noise(self, seeds, step):
        return torch.cat([_normal(sd, step, torch.arange(m, device=_DEV)) for sd, m in zip(seeds, self.local)])

    def step(self, step):
        self.f = self.forces()
        cs, sn = torch.cos(self.pol), torch.sin(self.pol)
        u = torch.stack([cs, sn], dim=1)[self.ring] + self.f  # vo = mobility = 1
        vx, vy = self.ring_sum(u[:, 0]) / self.np, self.ring_sum(u[:, 1]) / self.np
        cr = ((cs * vy - sn * vx) / torch.sqrt(vx * vx + vy * vy)).clamp(-1.0, 1.0)
        self.pos = self.space.wrap(self.pos + u * DT)
        self.pol = self.pol + torch.asin(cr) / RING["relax_time"] * DT + \
            math.sqrt(2 * RING["rot_diff"] * DT) * self.noise(self.seeds, step)

    def padded(self, v, base):
        """Per-particle rows into the (nrings * nmax, 2) layout; base holds the padding's values."""
        out = base.copy()
        out[self.mask[0].ravel()] = v.cpu().numpy()
        return out


def _net64(params, x):
    z, at = x, 0
    for k, (nout, nin) in enumerate(LAYERS):
        w = params[at:at + nout * nin].reshape(nout, nin)
        z = z @ w.T + params[at + nout * nin:at + nout * nin + nout]
        at += nout * nin + nout
        if k < 3:
            z = z * torch.sigmoid(1.702 * z)
    return z


def _learned_features(R, f, pol):
    """The propagator's 160 features per particle, in its ring's frame."""
    pos, sp = R.pos, R.space
    cs, sn = torch.cos(pol), torch.sin(pol)
    c, s = cs[R.ring], sn[R.ring]
    turn = lambda v: torch.stack([c * v[:, 0] + s * v[:, 1], -s * v[:, 0] + c * v[:, 1]], dim=1)  # noqa: E731
    u = torch.stack([c, s], dim=1) + f
    x = torch.zeros(len(pos), N_IN, dtype=F64, device=_DEV)
    x[:, 0] = R.type[R.ring].to(F64)
    x[:, 1] = ((R.areas - R.area0) / R.area0)[R.ring]
    x[:, 2:4], x[:, 4:6] = turn(R.diff(pos[R.prev], pos)), turn(R.diff(pos[R.next], pos))
    x[:, 6:8], x[:, 8:10], x[:, 10:12] = turn(u), turn(u[R.prev] - u), turn(u[R.next] - u)
    x[:, 12] = (R.ring_sum(u[:, 0] * R.da[:, 1] - u[:, 1] * R.da[:, 0]) / 2 / R.area0)[R.ring]
    vx, vy = R.ring_sum(u[:, 0]) / R.np, R.ring_sum(u[:, 1]) / R.np
    x[:, 13] = torch.asin(((cs * vy - sn * vx) / torch.sqrt(vx * vx + vy * vy)).clamp(-1.0, 1.0))[R.ring]
    js, oks = zip(*sp.blocks(sp.bins(pos)))
    j, ok = torch.cat(js, 1), torch.cat(oks, 1)
    dx, dy = sp.image(pos[j, 0] - pos[:, 0, None], pos[j, 1] - pos[:, 1, None])
    d2 = torch.where(ok, dx * dx + dy * dy, 1e30)
    d2 = torch.where(d2 <= R_FEAT * R_FEAT, d2, 1e30)
    d2, order = torch.sort(d2, dim=1, stable=True)
    m = min(32, d2.shape[1])
    d2, order = d2[:, :m], order[:, :m]
    j, dx, dy = (torch.gather(v, 1, order) for v in (j, dx, dy))
    near = d2 < 1e29
    rdot = ((u[j, 0] - u[:, 0, None]) * dx + (u[j, 1] - u[:, 1, None]) * dy) / torch.sqrt(d2)
    same = torch.where(R.ring[j] == R.ring[:, None], 1.0, -1.0)
    g = torch.stack([c[:, None] * dx + s[:, None] * dy, -s[:, None] * dx + c[:, None] * dy, same, rdot], dim=2)
    x[:, 32:32 + 4 * m] = (g * near[:, :, None]).reshape(len(pos), 4 * m)
    return x, u


def _learned_exact(case, seed):
    """Learned steps, all accepted (the listed and drawn states stay inside the gate)."""
    d = _ring_inputs(case, seed, R_FEAT)
    R, params = _Rings([d], [seed]), _t(_net_params(seed))
    kdt = K_PLAIN * DT
    for m in range(case["steps"]):
        f = R.forces()
        x, u = _learned_features(R, f, R.pol)
        y = _net64(params, x) * S_T
        cs, sn = torch.cos(R.pol), torch.sin(R.pol)
        c, s = cs[R.ring], sn[R.ring]
        disp = kdt * u + torch.stack([c * y[:, 0] - s * y[:, 1], s * y[:, 0] + c * y[:, 1]], dim=1)
        vx, vy = R.ring_sum(disp[:, 0]) / (R.np * kdt), R.ring_sum(disp[:, 1]) / (R.np * kdt)
        cr = ((cs * vy - sn * vx) / torch.sqrt(vx * vx + vy * vy)).clamp(-1.0, 1.0)
        R.pos = R.space.wrap(R.pos + disp)
        R.pol = R.pol + kdt / RING["relax_time"] * torch.asin(cr) + \
            math.sqrt(2 * RING["rot_diff"] * kdt) * R.noise([seed], K_PLAIN * m)
    return dict(pos=R.pos, pol=R.pol)


def _mix64(z):
    z = z + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _train_exact(case, seed):
    _, x, t = _train_inputs(case, seed)
    x, t = _t(x), _t(t.astype(np.float64))
    p = _t(_net_params(seed)).requires_grad_(True)
    m1, m2, losses = torch.zeros_like(p), torch.zeros_like(p), []
    row = np.arange(case["batch"], dtype=np.uint64)
    for s in range(case["steps"]):
        pick = _mix64(np.uint64(seed) ^ _mix64((np.uint64(s) << np.uint64(32)) ^ row)) % np.uint64(case["rows"])
        at = _t(pick.astype(np.int64), torch.int64)
        loss = ((_net64(p, x[at]) - t[at]) ** 2).sum() / (2 * case["batch"])
        g, = torch.autograd.grad(loss, p)
        m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
        step = 1e-3 * (m1 / (1 - 0.9 ** (s + 1))) / (torch.sqrt(m2 / (1 - 0.999 ** (s + 1))) + 1e-8)
        p = (p - step).detach().requires_grad_(True)
        losses.append(loss.detach())
    return dict(losses=torch.stack(losses), params=p.detach())


def exact(case, seed):
    with torch.no_grad() if case["family"] != "train" else torch.enable_grad():
        family, steps = case["family"], case["steps"]
        if family == "train":
            return _train_exact(case, seed)
        if family == "learned":
            out = _learned_exact(case, seed)
        elif family == "active":
            out = _active_exact(case, seed)
        elif family == "gas":
            d = _gas_inputs(case, seed)
            space = _Space([dict(d, n=len(d["pos"]))], case["walls"] == "periodic")
            law = {"lj": _lj(2.5), "lj_ref": _lj(math.inf), "harm": _harm(HARM)}[case["potential"]]
            radius = 2 ** (1 / 6) / 2 if case["potential"] != "harm" else HARM["dist_eq"] / 2
            pos, vel = _t(d["pos"]), _t(d["vel"])
            for _ in range(steps):
                pos, vel, f = _verlet_step(space, pos, vel, law, radius)
            out = dict(pos=pos, forces=f, vel=vel)
        elif family == "rings":
            d = _ring_inputs(case, seed)
            R = _Rings([d], [seed])
            for k in range(steps):
                R.step(k + 1)
            flat = d["pos"].reshape(-1, 2)
            out = dict(pos=R.padded(R.pos, flat), forces=R.padded(R.f, np.zeros_like(flat)), pol=R.pol, areas=R.areas)
        else:
            parts = _batch_inputs(case, seed)
            gas = [d for kind, d in parts if kind == "gas"]
            ring = [d for kind, d in parts if kind == "rings"]
            space = _Space([dict(d, n=len(d["pos"])) for d in gas])
            pos, vel = (_t(np.concatenate([d[k] for d in gas])) for k in ("pos", "vel"))
            R = _Rings(ring, [seed + i for i, (kind, _) in enumerate(parts) if kind == "rings"])
            for k in range(steps):
                pos, vel, _ = _verlet_step(space, pos, vel, _lj(2.5), 0.0)
                R.step(k + 1)
            at, rt, rows = 0, 0, []
            for kind, d in parts:  # the replicas in turn again (full rings: no padding)
                n = d["pos"].size // 2
                src, o = (pos, at) if kind == "gas" else (R.pos, rt)
                rows.append(src[o:o + n])
                at, rt = (at + n, rt) if kind == "gas" else (at, rt + n)
            out = dict(pos=torch.cat(rows), vel=vel, pol=R.pol)
        return {k: v if isinstance(v, np.ndarray) else v.cpu() for k, v in out.items()}
