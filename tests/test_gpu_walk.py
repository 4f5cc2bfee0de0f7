"""Pair sets of the home-cell walk at the sizes where it can go wrong: less than a
wavefront, exactly one and one more particle per cell, a cell more crowded than one
window of candidates, boxes too short for the home frame, open axes, exclusion rows
longer than the four kept in registers, and asymmetric rows; all against the oracle's
pairlist (bit for bit the same set)."""
import numpy as np
import pytest

import marsmd
from marsmd import configs
from marsmd.core import ExclusionCSR, PeriodicBox
from oracle import pyoracle as orc
from tests.conftest import sorted_pairs

pytestmark = pytest.mark.gpu


def _system(n, L, crowd, seed):
    rs = np.random.default_rng(seed)
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = rs.uniform(0, L, size=(n, 3))
    k = min(crowd, n)  # beads crowded into a corner of the box, across its seams
    pos[:k, :3] = np.mod(rs.uniform(-1.5, 1.5, size=(k, 3)), L)
    return pos


# (beads, box, cutoff, beads crowded into one corner)
SHAPES = [(1, 60.0, 9.0, 0), (2, 60.0, 9.0, 2), (63, 60.0, 9.0, 63), (64, 60.0, 9.0, 64), (65, 60.0, 9.0, 65),
          (700, 40.0, 18.0, 0), (1500, 90.0, 10.0, 130), (6000, 400.0, 12.0, 3000), (20011, 200.0, 10.0, 40)]


@pytest.mark.parametrize("periodic", [(True, True, True), (False, True, False)])
@pytest.mark.parametrize("shape", SHAPES)
def test_pair_sets(cuda, shape, periodic):
    n, L, rc, crowd = shape
    pos = _system(n, L, crowd, 7 * n + crowd)
    box = PeriodicBox((L, L * 1.1, L * 0.9), periodic=periodic)
    pos[:, 2] = np.minimum(pos[:, 2], np.nextafter(np.float32(L * 0.9), np.float32(0)))
    print("case:", shape, periodic, flush=True)
    pl = marsmd.create_pairlist(n)
    pl.set_periodic_box(box)
    pl.build_pairlist(cuda.from_numpy(pos).cuda(), n, rc)
    got = sorted_pairs(pl.get_neighbor_pairs().cpu().numpy())
    assert np.array_equal(got, orc.build_pairlist(pos, box, rc)["pairs"].astype(np.int64))


@pytest.mark.parametrize("symmetric", [True, False])
def test_long_exclusion_rows_of_a_caller(cuda, symmetric):
    # rows of 0..7 entries; asymmetric: only the lower sorted index's row counts
    n, L, rc = 3000, 70.0, 11.0
    pos = _system(n, L, 90, 3)
    box = PeriodicBox((L, L, L))
    rs = np.random.default_rng(4)
    near = orc.build_pairlist(pos, box, rc)["pairs"]
    ex = near[rs.permutation(len(near))[:5000]]
    off, exc, ne = marsmd.exclusion_csr_from_pairs(ex)
    if not symmetric:  # every other entry of every row stays
        rows = [exc[off[i]:off[i + 1]][::2] for i in range(ne)]
        off = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
        exc = np.concatenate(rows).astype(np.int32)
    view = ExclusionCSR(offsets=cuda.from_numpy(off).cuda(), excluded=cuda.from_numpy(exc).cuda(), num_particles=ne)
    pl = marsmd.create_pairlist(n)
    pl.set_periodic_box(box)
    pl.set_exclusions(view)
    pl.build_pairlist(cuda.from_numpy(pos).cuda(), n, rc)
    got = sorted_pairs(pl.get_neighbor_pairs().cpu().numpy())
    ref = orc.build_pairlist(pos, box, rc, offsets=off, excluded=exc, num_excl=ne)
    assert np.array_equal(got, ref["pairs"].astype(np.int64))


@pytest.mark.parametrize("L", [120.0, 420.0])  # with and without the home frame
def test_patch_exclusions_longer_than_the_registers(cuda, L):
    spec = configs.config1(chains=12, beads=60, L=L, seed=5)
    idx = np.arange(720).reshape(12, 60)
    extra = [np.stack([idx[:, :-k].ravel(), idx[:, k:].ravel()], axis=1) for k in (3, 4, 5)]
    spec.exclusions = np.vstack([spec.exclusions, *extra]).astype(np.int32)
    patch, sim = marsmd.Patch(spec), orc.Sim(spec)
    patch.run(1)
    sim.run(1)
    got = sorted_pairs(patch.get_pairlist().get_neighbor_pairs().cpu().numpy())
    assert np.array_equal(got, sorted_pairs(sim.get_pairs()))
