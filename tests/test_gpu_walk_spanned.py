"""Pair sets of the walk in boxes that the list cutoff spans on one, two or all axes, at the
sizes and shapes where its cells are chosen another way, against the oracle's pairlist; and
the bits of replicas in such boxes, alone and beside others."""
import dataclasses

import numpy as np
import pytest

import marsmd
from marsmd import configs
from marsmd.batch import Batch
from marsmd.core import PeriodicBox
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu

# one axis, two axes, three axes spanned; the home frame at no level, at the next finer one
SHAPES = [(5000, (200.0, 200.0, 60.0), 28.0), (20000, (300.0, 300.0, 40.0), 19.0), (1000, (300.0, 40.0, 40.0), 18.0),
          (6000, (30.0, 150.0, 30.0), 14.0), (20000, (200.0, 200.0, 30.0), 12.2), (20000, (200.0, 200.0, 30.0), 13.9),
          (30011, (500.0, 300.0, 45.0), 22.0), (2000, (80.0, 80.0, 80.0), 29.0), (500, (60.0, 60.0, 60.0), 25.0),
          (9000, (90.0, 100.0, 110.0), 40.0), (16384, (80.0, 80.0, 80.0), 34.0), (16385, (80.0, 80.0, 80.0), 34.0)]


def _mixed(key):
    """A number per pair whose sum tells pair sets apart (wrapping int64, numpy or torch)."""
    k = key * -7046029254386353131
    return ((k ^ (k >> 29)) * -4658895280553007687).sum()


@pytest.mark.parametrize("shape", SHAPES)
def test_pair_sets(cuda, shape):
    n, L, rc = shape
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = np.random.default_rng(n).uniform(0, 1, (n, 3)) * L
    pos[:, :3] = np.minimum(pos[:, :3], np.nextafter(np.float32(L), np.float32(0)))
    box = PeriodicBox(L)
    print("case:", shape, flush=True)
    pl = marsmd.create_pairlist(n)
    pl.set_periodic_box(box)
    pl.build_pairlist(cuda.from_numpy(pos).cuda(), n, rc)
    got = pl.get_neighbor_pairs().long()
    ref = orc.build_pairlist(pos, box, rc)["pairs"].astype(np.int64)
    assert len(got) == len(ref)
    lo, hi = cuda.minimum(got[:, 0], got[:, 1]), cuda.maximum(got[:, 0], got[:, 1])
    with np.errstate(over="ignore"):
        want = int(_mixed(ref.min(axis=1) * n + ref.max(axis=1)))
    assert int(_mixed(lo * n + hi)) == want


def test_replicas_keep_their_bits(cuda):
    specs = []
    for r, (n, L, _) in enumerate(SHAPES[:2] + SHAPES[4:5] + SHAPES[7:10]):
        s = configs.config3(replicas=1, n_min=n, n_max=n, density=4e-4, seed=29)[0]
        s.box = PeriodicBox(L)
        s.positions = (np.random.default_rng(r).uniform(0, 0.999, (n, 3)) * L).astype(np.float32)
        specs.append(dataclasses.replace(s, patch_id=r, params=dataclasses.replace(
            s.params, cutoff=10.0, pairlist_cutoff=12.2, timestep=s.params.timestep / 1e4, rebuild_period=5)))
    for s in specs[:1] + specs[3:]:  # a cutoff that spans their boxes
        print("case:", s.n, s.box.size, flush=True)
    for rc in (12.2, 28.0):
        for s in specs:
            s.params = dataclasses.replace(s.params, cutoff=rc - 2.0, pairlist_cutoff=rc)
        few = specs if rc < 20.0 else [specs[0]] + specs[3:]
        b = Batch(few)
        b.run(7)
        for s, got in zip(few, b.copy_particles_to_host()):
            one = Batch([s])
            one.run(7)
            alone = one.copy_particles_to_host()[0]
            for k in ("pos", "force", "id"):
                assert np.array_equal(got[k], alone[k]), f"{k} of {s.n} beads at cutoff {rc}"
