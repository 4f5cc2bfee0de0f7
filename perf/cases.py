"""The work that programs have this library do, as cases with their inputs, one pass
through the public entry points, its cost and its tolerance.

A simulation program advances a system by some steps and takes the frame; a scoring or
output step evaluates forces and energies through the separate calls; replicas advance
together as a batch; a fit of pair tables evaluates its loss and gradient over snapshots;
a program with its own integrator builds a pairlist over device arrays and launches the
pair kernel on it. Sizes run from a few hundred beads (latency) to a million.

The simulations keep their particle labels for 1000 steps (reorder_period) so that the
rows of consecutive frames line up; the pairlist is checked every 20 steps as usual.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mars-md_amd"))

import marsmd  # noqa: E402
from marsmd import _capi as api  # noqa: E402
from marsmd import configs  # noqa: E402
from marsmd.batch import Batch  # noqa: E402
from marsmd.core import Grid, PairParams, ParticleType, PeriodicBox, make_pair_tag  # noqa: E402
from marsmd.fm import ForceMatching, force_matching_loss  # noqa: E402
from marsmd.system import RunParams, SystemSpec  # noqa: E402

CUTOFF, LIST_CUTOFF = 30.0, 35.0
PERIOD = 20  # steps between pairlist checks
REORDER = 1000
DT, KT = 1e-4, 0.593
MIN_SEPARATION = 3.0


# ------------------------------------------------------------------------- the cases
def listed():
    return [
        # one small solute system, as a parameter scan runs thousands of: launches and latency
        {"name": "beads-500", "kind": "beads", "n": 500, "density": 1e-4, "steps": 100},
        # the plain Brownian system of the framework's first workload (L = 250 A)
        {"name": "beads-10k", "kind": "beads", "n": 10_000, "density": 6.4e-4, "steps": 100},
        # an ordinary mid-size system, no round number of tiles
        {"name": "beads-100003", "kind": "beads", "n": 100_003, "density": 1e-4, "steps": 100},
        # bead-spring polymers: bonds, angles, exclusions, very uneven neighbour counts
        {"name": "polymers-200x500", "kind": "polymers", "chains": 200, "beads": 500, "density": 1.953e-4, "steps": 40},
        # Langevin beads in a trilinearly sampled field on a ragged grid
        {"name": "field-60001-linear", "kind": "field", "n": 60_001, "density": 1.25e-4, "grid": 97, "cubic": False,
         "steps": 100},
        # the headline: a million Langevin beads, 256^3 tricubic membrane field
        {"name": "field-1m-cubic", "kind": "field", "n": 1_000_000, "density": 1.25e-4, "grid": 256, "cubic": True,
         "steps": 100},
        # energy output at every step through the separate calls; tables plus screened charges
        {"name": "energies-30011", "kind": "energies", "n": 30_011, "density": 4e-4, "steps": 20},
        # a handful of replicas (umbrella windows), and the large replica batch
        {"name": "batch-24", "kind": "batch", "replicas": 24, "n_min": 500, "n_max": 4_000, "steps": 100},
        {"name": "batch-512", "kind": "batch", "replicas": 512, "n_min": 500, "n_max": 20_000, "steps": 100},
        # force matching: a quick fit on a few small snapshots, and the full data set
        {"name": "fit-5x7001", "kind": "fit", "snapshots": 5, "n": 7_001, "density": 1e-4, "knots": 512},
        {"name": "fit-64x100k", "kind": "fit", "snapshots": 64, "n": 100_000, "density": 1e-4, "knots": 512},
        # a caller with its own arrays: pairlist build, pairs, tags, pair forces
        {"name": "pairs-80021", "kind": "pairs", "n": 80_021, "density": 2e-4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["beads", "polymers", "field", "energies", "batch", "fit", "pairs"])
    steps = 20 * rng.randint(1, 5)
    density = math.exp(rng.uniform(math.log(1e-4), math.log(6.4e-4)))
    if kind == "beads":
        return {"kind": kind, "n": _log(rng, 500, 250_000), "density": density, "steps": steps}
    if kind == "polymers":
        return {"kind": kind, "chains": _log(rng, 5, 220), "beads": rng.randint(60, 500), "density": 1.953e-4,
                "steps": min(steps, 40)}
    if kind == "field":
        return {"kind": kind, "n": _log(rng, 2_000, 900_000), "density": 1.25e-4, "grid": rng.randint(40, 256),
                "cubic": rng.random() < 0.6, "steps": steps}
    if kind == "energies":
        return {"kind": kind, "n": _log(rng, 600, 150_000), "density": density, "steps": 20}
    if kind == "batch":
        return {"kind": kind, "replicas": _log(rng, 3, 400), "n_min": 500, "n_max": _log(rng, 700, 20_000),
                "steps": steps}
    if kind == "fit":
        return {"kind": kind, "snapshots": _log(rng, 2, 40), "n": _log(rng, 1_500, 100_000), "density": 1e-4,
                "knots": rng.choice([256, 301, 512])}
    return {"kind": kind, "n": _log(rng, 1_000, 200_000), "density": density}


# ------------------------------------------------------------------------- inputs
def _positions(n, L, r):
    """Beads on distinct random sites of a fine lattice, displaced at random within the
    site less the minimum separation."""
    m = max(int(L // (2 * MIN_SEPARATION)), 1)
    if m ** 3 < 2 * n:
        raise ValueError("too dense")
    s = r.choice(m ** 3, n, replace=False, shuffle=False)
    r.shuffle(s)
    h = L / m
    site = np.stack([s // (m * m), (s // m) % m, s % m], axis=1).astype(np.float64)
    p = (site + 0.5 + r.uniform(-0.5, 0.5, (n, 3)) * (1.0 - MIN_SEPARATION / h)) * h
    return np.clip(p, 0.0, np.nextafter(np.float32(L), np.float32(0.0))).astype(np.float32)


def _chains(chains, beads, L, r):
    """Walks of 5 A steps with the stiffness that the angle potential gives at kT (a mean
    cosine of about 0.7 between steps), as relaxed chains have it."""
    t = r.standard_normal((chains, 3))
    t /= np.linalg.norm(t, axis=1, keepdims=True)
    p = np.empty((chains, beads, 3))
    p[:, 0] = r.uniform(0.0, L, (chains, 3))
    for b in range(1, beads):
        t += 0.55 * r.standard_normal((chains, 3))
        t /= np.linalg.norm(t, axis=1, keepdims=True)
        p[:, b] = p[:, b - 1] + 5.0 * t
    p = np.mod(p.reshape(-1, 3), L)
    return np.clip(p, 0.0, np.nextafter(np.float32(L), np.float32(0.0))).astype(np.float32)


def _params(**kw):
    return RunParams(**{**dict(cutoff=CUTOFF, pairlist_cutoff=LIST_CUTOFF, rebuild_period=PERIOD,
                               reorder_period=REORDER, timestep=DT, kT=KT), **kw})


def _box_length(n, density):
    return float((n / density) ** (1.0 / 3.0))


def _beads(n, density, r, seed, patch_id=0):
    L = _box_length(n, density)
    return SystemSpec(box=PeriodicBox((L, L, L)), types=[ParticleType(diffusion=(150.0,) * 3)],
                      positions=_positions(n, L, r), type_ids=np.zeros(n, np.int32), params=_params(),
                      nb_tables=[configs.pair_table(qq=1.0)], seed=seed, patch_id=patch_id)


def _spec(case, seed):
    r = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "beads":
        return _beads(case["n"], case["density"], r, seed)
    if kind == "polymers":
        n = case["chains"] * case["beads"]
        L = _box_length(n, case["density"])
        spec = configs.config1(chains=case["chains"], beads=case["beads"], L=L, seed=seed)
        spec.positions = _chains(case["chains"], case["beads"], L, r)
        spec.params = _params()
        return spec
    n = case["n"]
    L = _box_length(n, case["density"])
    if kind == "field":
        q = [1.0, -1.0, 0.5]
        mass, gamma = 100.0, 1000.0
        pairs = [(i, j) for i in range(3) for j in range(i, 3)]
        tags = np.zeros((3, 3), np.uint32)
        for k, (i, j) in enumerate(pairs):
            tags[i, j] = tags[j, i] = make_pair_tag(api.PAIR_TERM_TABULATED, k)
        return SystemSpec(
            box=PeriodicBox((L, L, L)),
            types=[ParticleType(mass=mass, charge=c, diffusion=(KT / (mass * gamma),) * 3, trans_damping=(gamma,) * 3,
                                pmf_terms=[(0, c, -1)]) for c in q],
            positions=_positions(n, L, r), type_ids=r.integers(0, 3, n).astype(np.int32),
            momenta=(math.sqrt(KT * mass) * configs.SQRT_CAL_TO_JOULE * r.standard_normal((n, 3), np.float32)),
            params=_params(integrator=api.INTEGRATOR_LANGEVIN,
                           interpolation=api.INTERP_CUBIC if case["cubic"] else api.INTERP_LINEAR),
            nb_tables=[configs.pair_table(qq=q[i] * q[j]) for i, j in pairs], term_matrix=tags,
            grids=[configs.membrane_grid(L, case["grid"])], seed=seed)
    # energies: a repulsive table for all pairs, screened charges from the analytical term
    q = [0.5, -0.5]
    tags = np.full((2, 2), make_pair_tag(api.PAIR_TERM_TABULATED | api.PAIR_TERM_DEBYE_HUCKEL, 0), np.uint32)
    return SystemSpec(
        box=PeriodicBox((L, L, L)), types=[ParticleType(charge=c, diffusion=(150.0,) * 3) for c in q],
        positions=_positions(n, L, r), type_ids=r.integers(0, 2, n).astype(np.int32),
        params=_params(energy_period=1), nb_tables=[configs.pair_table(qq=0.0)], term_matrix=tags,
        enabled_terms=api.PAIR_TERM_TABULATED | api.PAIR_TERM_DEBYE_HUCKEL, pair_params=PairParams(), seed=seed)


def _replicas(case, seed):
    r = np.random.default_rng(seed)
    k = case["replicas"]
    # sizes spread evenly over their logarithm, in no order
    u = (r.permutation(k) + 0.5) / k
    ns = np.round(np.exp(np.log(case["n_min"]) + u * np.log(case["n_max"] / case["n_min"]))).astype(int)
    return [_beads(int(n), 1e-4, r, seed, patch_id=i) for i, n in enumerate(ns)]


def _fit(case, seed):
    r = np.random.default_rng(seed)
    n, S = case["n"], case["snapshots"]
    L = _box_length(n, case["density"])
    tables, tags = configs.fm_tables(case["knots"])
    pos = np.stack([_positions(n, L, r) for _ in range(S)])
    types = r.integers(0, 4, n).astype(np.int32)
    start = configs.perturbed_tables(tables, 0.2, seed)
    target = 2.0 * r.standard_normal((S, n, 3), np.float32)  # fitted forces, kcal/mol/A
    return L, tables, tags, pos, types, start, target


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("beads", "polymers", "field", "energies"):
        spec = _spec(case, seed)
        return {"kind": kind, "steps": case["steps"], "step": 0, "spec": spec, "patch": marsmd.Patch(spec)}
    if kind == "batch":
        specs = _replicas(case, seed)
        return {"kind": kind, "steps": case["steps"], "step": 0, "batch": Batch(specs)}
    if kind == "fit":
        L, tables, tags, pos, types, start, target = _fit(case, seed)
        fm = ForceMatching(pos, types, PeriodicBox((L, L, L)), tables, tags, CUTOFF)
        return {"kind": kind, "fm": fm, "knots": fm.knots(start).requires_grad_(True),
                "target": torch.from_numpy(target).cuda()}
    spec = _spec({**case, "kind": "energies"}, seed)
    pl = marsmd.create_pairlist(spec.n)
    pl.set_periodic_box(spec.box)
    return {"kind": kind, "spec": spec, "pairlist": pl, "pos": torch.from_numpy(spec.pos4()).cuda(),
            "types": torch.from_numpy(spec.type_ids).cuda(), "tables": marsmd.DeviceTables(spec.nb_tables),
            "tags": torch.from_numpy(spec.tag_matrix().view(np.int32)).cuda()}


# ------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind in ("beads", "polymers", "field"):
        patch = state["patch"]
        patch.run(state["steps"], first_step=state["step"])
        state["step"] += state["steps"]
        h = patch.copy_particles_to_host()
        frame = {"pos": h["pos"], "id": h["id"]}
        if kind == "field":
            frame["mom"] = h["mom"]
        return frame
    if kind == "energies":
        patch = state["patch"]
        for _ in range(state["steps"]):
            state["step"] += 1
            patch.step_unfused(state["step"])
        h = patch.copy_particles_to_host()
        return {"pos": h["pos"], "force_energy": h["force"], "id": h["id"]}
    if kind == "batch":
        batch = state["batch"]
        batch.run(state["steps"], first_step=state["step"])
        state["step"] += state["steps"]
        return {"pos": np.concatenate([h["pos"] for h in batch.copy_particles_to_host()])}
    if kind == "fit":
        knots = state["knots"]
        knots.grad = None
        loss = force_matching_loss(knots, state["fm"], state["target"])
        loss.backward()
        return {"loss": loss.detach(), "grad": knots.grad}
    spec, pos = state["spec"], state["pos"]
    pl = state["pairlist"]
    pl.build_pairlist(pos, spec.n, LIST_CUTOFF)
    pairs = pl.get_neighbor_pairs()
    num = pl.get_num_pairs()
    tag = torch.empty(num, dtype=torch.int32, device="cuda")
    marsmd.launch_resolve_pair_tables(pairs, state["types"], state["tags"], 2, tag, num)
    force = torch.zeros(spec.n, 4, device="cuda")
    view = marsmd.particle_view(pos=pos, force_energy=force, type_id=state["types"])
    marsmd.launch_pairwise_nonbonded(pairs, view, tag, state["tables"], spec.box, True, num, CUTOFF * CUTOFF,
                                     enabled_terms=spec.enabled_terms, types=spec.types, params=spec.pair_params)
    return {"force_energy": force, "pairs": num}


# ------------------------------------------------------------------------- cost
def _mean_beads(case):
    ratio = case["n_max"] / case["n_min"]
    return case["n_min"] if ratio == 1 else (case["n_max"] - case["n_min"]) / math.log(ratio)


def work(case):
    """Per step: positions read and written once, momenta too, the field once, the
    topology once; per list life the list written once and per step read once (4 bytes a
    half pair); the arithmetic of the pairs within the cutoff, of the field's taps and of
    the integrator. A frame is written once."""
    kind = case["kind"]
    sphere = 4.0 / 3.0 * math.pi
    if kind == "fit":
        half = 0.5 * sphere * CUTOFF ** 3 * case["density"]
        rows = case["snapshots"] * case["n"]
        return {"bytes": rows * (16 + 12 + 4 * half) + 10 * case["knots"] * 12, "flops": rows * half * 2 * 40}
    if kind == "batch":
        n, density = case["replicas"] * _mean_beads(case), 1e-4
    elif kind == "polymers":
        n, density = case["chains"] * case["beads"], case["density"]
    else:
        n, density = case["n"], case["density"]
    half_list = 0.5 * sphere * LIST_CUTOFF ** 3 * density
    half = 0.5 * sphere * CUTOFF ** 3 * density
    if kind == "pairs":
        return {"bytes": n * (16 + 16 + 4 + 12 * half_list), "flops": n * half * 40}
    state = 32.0
    flops = 40 * half + 60
    if kind == "polymers":
        state += 8 + 12
        flops += 150
    if kind == "field":
        state += 32 + 4.0 * case["grid"] ** 3 / n
        flops += 300 if case["cubic"] else 60
    if kind == "energies":
        state += 16
    steps = case["steps"]
    return {"bytes": n * (steps * (state + 4 * half_list * (1 + 1 / PERIOD)) + 32), "flops": n * steps * flops}


# ------------------------------------------------------------------------- tolerance
def tolerance(case):
    """Measured with the force sums in another order (other walk cells: positions within
    2e-6 after 80 steps of polymers and 1e-8 otherwise, momenta 2e-7) and against the
    64-bit reference (positions 1e-5, momenta 3e-3, forces at the last step 8e-3, pair
    forces of given positions 7e-6), stated in between. A table's force jumps from bin to
    bin, so where a distance moved by rounding crosses a knot one pair's force changes by
    some percent, and a collision multiplies what it meets: hence the room for single
    values."""
    return {"beads": {"rel": 1e-5, "max": 1e-2}, "batch": {"rel": 1e-5, "max": 1e-2},
            "polymers": {"rel": 2e-5, "max": 2e-2}, "field": {"rel": 3e-4, "max": 0.5},
            "energies": {"rel": 2e-3, "max": 0.5}, "fit": {"rel": 1e-5, "max": 1e-3},
            "pairs": {"rel": 2e-5, "max": 1e-2}}[case["kind"]]


# ------------------------------------------------------------------------- 64-bit reference
F64 = torch.float64


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _f32(x):
    """The value a 32-bit parameter holds."""
    return float(np.float32(x))


def _min_image(d, L):
    return d - L * torch.round(d / L)


def _close_pairs(x, L, rc):
    """Every pair (i, j) of `x` within rc in a periodic cube, once."""
    n, nc = len(x), int(L // rc)
    dev = x.device
    if nc < 3:
        i, j = torch.triu_indices(n, n, 1, device=dev)
        keep = _min_image(x[j] - x[i], L).square().sum(1) <= rc * rc
        return i[keep], j[keep]
    c = torch.clamp((x / L * nc).floor().long(), 0, nc - 1)
    order = torch.argsort((c[:, 0] * nc + c[:, 1]) * nc + c[:, 2])
    c, xs = c[order], x[order]
    count = torch.bincount((c[:, 0] * nc + c[:, 1]) * nc + c[:, 2], minlength=nc ** 3)
    start = torch.cumsum(count, 0) - count
    me = torch.arange(n, device=dev)
    out_i, out_j = [], []
    half = [(a, b, d) for a in (-1, 0, 1) for b in (-1, 0, 1) for d in (-1, 0, 1) if (a, b, d) >= (0, 0, 0)]
    for o in half:
        k = (c + torch.tensor(o, device=dev)) % nc
        k = (k[:, 0] * nc + k[:, 1]) * nc + k[:, 2]
        m = count[k]
        i = torch.repeat_interleave(me, m)
        j = torch.arange(len(i), device=dev) - (torch.cumsum(m, 0) - m)[i] + start[k][i]
        if o == (0, 0, 0):
            keep = j > i
            i, j = i[keep], j[keep]
        keep = _min_image(xs[j] - xs[i], L).square().sum(1) <= rc * rc
        out_i.append(order[i[keep]])
        out_j.append(order[j[keep]])
    return torch.cat(out_i), torch.cat(out_j)


def _table(U, step_inv, d):
    """-dU/dr (constant within a bin) and U of a table on [0, last knot] at distances d;
    U is one table (knots,) or one per pair of d through a flat array and offsets."""
    knots, base = U
    size = knots.shape[-1]
    w = d * step_inv
    h = w.floor().long()
    beyond = h >= size - 1
    h = h.clamp(0, size - 2)
    flat = knots.reshape(-1)
    at = h + base * size
    U0, U1 = flat[at], flat[at + 1]
    return torch.where(beyond, 0.0, -(U1 - U0) * step_inv), torch.where(beyond, U1, (U1 - U0) * (w - h) + U0)


class _Exact:
    """The system of a spec stepped in 64 bits."""

    def __init__(self, spec):
        dev = _dev()
        t = lambda a, k=F64: torch.as_tensor(np.asarray(a), dtype=k, device=dev)  # noqa: E731
        self.spec, self.P, self.dev, self.n = spec, spec.params, dev, spec.n
        self.L = _f32(spec.box.size[0])
        self.x = t(spec.positions)[:, :3].clone()
        self.ty = t(spec.type_ids, torch.int64)
        self.mom = None if spec.momenta is None else t(spec.momenta).clone()
        self.knots = t(np.stack([u.pot for u in spec.nb_tables]))
        self.step_inv = spec.nb_tables[0].step_inv
        self.table_of = t(spec.tag_matrix().astype(np.int64) >> api.PAIR_TABLE_SHIFT, torch.int64)
        self.dh = bool(spec.enabled_terms & api.PAIR_TERM_DEBYE_HUCKEL)
        self.charge = t([p.charge for p in spec.types])[self.ty]
        self.grid = t(spec.grids[0].values) if spec.grids else None
        self.excluded = None
        if spec.exclusions is not None:
            e = np.sort(spec.exclusions.astype(np.int64), axis=1)
            self.excluded = torch.unique(t(e[:, 0] * spec.n + e[:, 1], torch.int64))
        if spec.bonds is not None:
            self.bonds = t(spec.bonds, torch.int64)
            self.angles = t(spec.angles, torch.int64)
            self.bond_U = t(spec.bond_tables[0].pot)
            self.angle_U = t(spec.angle_tables[0].pot)
        self.listed_at = None
        self.deferred = False

    def update_list(self, step):
        if (step - 1) % PERIOD:
            return
        if self.listed_at is not None:
            moved = _min_image(self.x - self.listed_at, self.L).square().sum(1).max()
            if moved <= (0.5 * (LIST_CUTOFF - CUTOFF)) ** 2:
                return
        i, j = _close_pairs(self.x, self.L, LIST_CUTOFF)
        if self.excluded is not None:
            key = torch.minimum(i, j) * self.n + torch.maximum(i, j)
            keep = ~torch.isin(key, self.excluded)
            i, j = i[keep], j[keep]
        self.i, self.j, self.listed_at = i, j, self.x.clone()

    def forces(self):
        """(n, 4) force and energy of the listed pairs within the cutoff and the bonded terms."""
        r = _min_image(self.x[self.j] - self.x[self.i], self.L)
        d = r.square().sum(1).sqrt()
        keep = (d <= CUTOFF) & (d >= 1e-6)
        i, j, r, d = self.i[keep], self.j[keep], r[keep], d[keep]
        f, u = _table((self.knots, self.table_of[self.ty[i], self.ty[j]]), self.step_inv, d)
        if self.dh:
            p = self.spec.pair_params
            e = self.charge[i] * self.charge[j] * _f32(332.0636) / p.dielectric * torch.exp(-d / p.debye_length) / d
            f, u = f + e * (1 / d + 1 / p.debye_length), u + e
        out = torch.zeros(self.n, 4, dtype=F64, device=self.dev)
        v = r * (f / d)[:, None]
        half = 0.5 * u[:, None]
        out.index_add_(0, j, torch.cat([v, half], 1))
        out.index_add_(0, i, torch.cat([-v, half], 1))
        if self.spec.bonds is not None:
            self.bonded(out)
        return out

    def bonded(self, out):
        a, b = self.bonds.T
        r = _min_image(self.x[b] - self.x[a], self.L)
        d = r.square().sum(1).sqrt()
        f, _ = _table((self.bond_U, 0), self.spec.bond_tables[0].step_inv, d)
        v = r * (f / d)[:, None]
        out[:, :3].index_add_(0, b, v)
        out[:, :3].index_add_(0, a, -v)
        a, b, c = self.angles.T
        ab, bc = _min_image(self.x[b] - self.x[a], self.L), _min_image(self.x[c] - self.x[b], self.L)
        lab, lbc = ab.square().sum(1).sqrt(), bc.square().sum(1).sqrt()
        ac = _min_image(self.x[c] - self.x[a], self.L)
        cos = ((lab ** 2 + lbc ** 2 - ac.square().sum(1)) * 0.5 / (lab * lbc)).clamp(-1.0, 1.0)
        # a periodic table of `size` knots over the angle in radians
        size, inv = len(self.angle_U), self.spec.angle_tables[0].step_inv
        h = (torch.acos(cos) * inv).floor().long() % size
        f = -(self.angle_U[(h + 1) % size] - self.angle_U[h]) * inv
        dU = (-f / torch.sqrt(1 - cos * cos).clamp(min=1e-3))[:, None]
        lab, lbc, cos = lab[:, None], lbc[:, None], cos[:, None]
        f1 = dU / lab * (cos / lab * ab + bc / lbc)
        f3 = -dU / lbc * (cos / lbc * bc + ab / lab)
        out[:, :3].index_add_(0, a, f1)
        out[:, :3].index_add_(0, b, -(f1 + f3))
        out[:, :3].index_add_(0, c, f3)

    def field(self):
        """Force of the periodic grid potential scaled by type."""
        n = self.grid.shape[0]
        inv = _f32(np.float32(1.0) / np.float32(self.spec.grids[0].spacing[0]))
        g = self.x * inv
        h = g.floor()
        t = g - h
        h = h.long()
        if self.P.interpolation == api.INTERP_CUBIC:
            first, w = -1, [0.5 * (2 * t ** 2 - t ** 3 - t), 0.5 * (3 * t ** 3 - 5 * t ** 2 + 2),
                            0.5 * (4 * t ** 2 - 3 * t ** 3 + t), 0.5 * (t ** 3 - t ** 2)]
            dw = [0.5 * (4 * t - 3 * t ** 2 - 1), 0.5 * (9 * t ** 2 - 10 * t), 0.5 * (8 * t - 9 * t ** 2 + 1),
                  0.5 * (3 * t ** 2 - 2 * t)]
        else:
            first, w, dw = 0, [1 - t, t], [-torch.ones_like(t), torch.ones_like(t)]
        flat = self.grid.reshape(-1)
        grad = torch.zeros_like(self.x)
        for a in range(len(w)):
            ox = (h[:, 0] + a + first) % n * (n * n)
            for b in range(len(w)):
                oxy = ox + (h[:, 1] + b + first) % n * n
                for c in range(len(w)):
                    v = flat[oxy + (h[:, 2] + c + first) % n]
                    grad[:, 0] += v * dw[a][:, 0] * w[b][:, 1] * w[c][:, 2]
                    grad[:, 1] += v * w[a][:, 0] * dw[b][:, 1] * w[c][:, 2]
                    grad[:, 2] += v * w[a][:, 0] * w[b][:, 1] * dw[c][:, 2]
        scale = torch.tensor([_f32(p.pmf_terms[0][1]) for p in self.spec.types], dtype=F64, device=self.dev)
        return grad * inv * -scale[self.ty][:, None]

    def noise(self, step, stream):
        """Box-Muller of the counter-based generator: key from the seed, the patch and the
        step, counter (particle, stream, step, 0)."""
        full = (1 << 64) - 1
        key = ((self.spec.seed * 0x9E3779B97F4A7C15) & full) ^ ((self.spec.patch_id << 32) & full)
        key ^= (step * 0xBF58476D1CE4E5B9) & full
        k0, k1, m = key >> 32, key & 0xFFFFFFFF, 0xFFFFFFFF
        word = lambda v: torch.full((self.n,), v, dtype=torch.int64, device=self.dev)  # noqa: E731
        c = [torch.arange(self.n, device=self.dev), word(stream), word(step), word(0)]
        for _ in range(10):
            p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
            c = [(p1 >> 32) & m ^ c[1] ^ k0, p1 & m, (p0 >> 32) & m ^ c[3] ^ k1, p0 & m]
            k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
        u = [v.to(F64) * 2.0 ** -32 + 2.0 ** -33 for v in c]
        r1, r2 = torch.sqrt(-2 * torch.log(u[0])), torch.sqrt(-2 * torch.log(u[2]))
        a1, a2 = 2 * math.pi * u[1], 2 * math.pi * u[3]
        return torch.stack([r1 * torch.cos(a1), r1 * torch.sin(a1), r2 * torch.cos(a2)], 1)

    def run(self, steps):
        P, dt, kT = self.P, _f32(self.P.timestep), _f32(self.P.kT)
        f = None
        for step in range(1, steps + 1):
            self.update_list(step)
            f = self.forces()
            if P.integrator == api.INTEGRATOR_BROWNIAN:
                D = _f32(self.spec.types[0].diffusion[0])
                self.x += D / kT * f[:, :3] * dt + math.sqrt(2 * D * dt) * self.noise(step, 0x5324120)
            else:
                kick = f[:, :3] + self.field() if self.grid is not None else f[:, :3]
                kick = 0.5 * dt * _f32(4.18679994e4) * kick
                mass, gamma = _f32(self.spec.types[0].mass), _f32(self.spec.types[0].trans_damping[0])
                a = math.exp(-gamma * dt)
                self.mom += 2 * kick if self.deferred else kick
                self.deferred = True
                drift = 0.5 * dt / mass * 10000.0
                self.x += drift * self.mom
                self.mom = a * self.mom + math.sqrt(kT * mass * (1 - a * a)) * _f32(2.046167337) * self.noise(step, 0x1356914)
                self.x += drift * self.mom
            self.x -= torch.floor(self.x / self.L) * self.L
        return f


def _rows4(v):
    return torch.nn.functional.pad(v, (0, 1)).cpu().numpy()


def _exact_fit(case, seed):
    L, tables, tags, pos, types, start, target = _fit(case, seed)
    dev = _dev()
    L = _f32(L)
    U = torch.tensor(np.stack([t.pot for t in start]), dtype=F64, device=dev)
    inv = tables[0].step_inv
    table_of = torch.tensor(tags.astype(np.int64) >> api.PAIR_TABLE_SHIFT, device=dev)
    ty = torch.tensor(types, dtype=torch.int64, device=dev)
    S, n = pos.shape[:2]
    loss, S_knot = 0.0, torch.zeros(U.numel(), dtype=F64, device=dev)
    for s in range(S):
        x = torch.tensor(pos[s], dtype=F64, device=dev)
        i, j = _close_pairs(x, L, CUTOFF)
        r = _min_image(x[j] - x[i], L)
        d = r.square().sum(1).sqrt()
        k = table_of[ty[i], ty[j]]
        h = (d * inv).floor().long()
        ok = h < U.shape[1] - 1
        i, j, r, d, k, h = i[ok], j[ok], r[ok], d[ok], k[ok], h[ok]
        u = r / d[:, None]
        at = k * U.shape[1] + h
        flat = U.reshape(-1)
        v = u * (-(flat[at + 1] - flat[at]) * inv)[:, None]
        f = torch.zeros(n, 3, dtype=F64, device=dev)
        f.index_add_(0, j, v)
        f.index_add_(0, i, -v)
        e = f - torch.tensor(target[s], dtype=F64, device=dev)
        loss += float(e.square().sum()) / (3.0 * S * n)
        G = e * (2.0 / (3.0 * S * n))
        g = ((G[j] - G[i]) * u).sum(1) * inv
        S_knot.index_add_(0, at, g)
        S_knot.index_add_(0, at + 1, -g)
    return {"loss": loss, "grad": S_knot.cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "fit":
        return _exact_fit(case, seed)
    if kind == "batch":
        if case["replicas"] > 60:  # one after another, too long
            return None
        frames = []
        for spec in _replicas(case, seed):
            e = _Exact(spec)
            e.run(case["steps"])
            frames.append(_rows4(e.x))
        return {"pos": np.concatenate(frames)}
    if kind == "pairs":
        e = _Exact(_spec({**case, "kind": "energies"}, seed))
        e.update_list(1)
        return {"force_energy": e.forces().cpu().numpy(), "pairs": len(e.i)}
    e = _Exact(_spec(case, seed))
    f = e.run(case["steps"])
    out = {"pos": _rows4(e.x), "id": None}
    if kind == "field":
        out["mom"] = _rows4(e.mom)
    if kind == "energies":
        out["force_energy"] = f.cpu().numpy()
    return out
