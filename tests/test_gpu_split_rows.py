"""Rows dealt to several lanes (8, 4 or 1 by the slot count): forces and steps against the
oracle where a round, a wavefront or a workgroup is not full, and the same bits on both
sides of each limit of the rule."""
import numpy as np
import pytest

import marsmd
from marsmd import _capi as api
from marsmd import configs
from oracle import pyoracle as orc
from tests.conftest import rel_force_error

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,L", [(1, 80.0), (7, 80.0), (33, 90.0), (64, 90.0), (129, 90.0), (1000, 140.0), (4001, 200.0)])
@pytest.mark.parametrize("cubic", [False, True])
def test_forces_and_steps_match_the_oracle(cuda, n, L, cubic):
    spec = configs.config2(n=n, L=L, grid_n=24, seed=n)
    spec.params.interpolation = api.INTERP_CUBIC if cubic else api.INTERP_LINEAR
    P = spec.params
    print("case:", n, L, cubic, flush=True)
    patch, sim = marsmd.Patch(spec), orc.Sim(spec)
    args = (P.pairlist_cutoff, P.cutoff, 1, P.rebuild_period)
    patch.calculate_nonbonded_forces(*args, compute_energy=True)
    sim.calculate_nonbonded_forces(*args, compute_energy=True)
    got, ref = patch.copy_particles_to_host(), sim.copy_particles_to_host()
    if np.abs(ref["force64"]).max() > 0:
        assert rel_force_error(got["force"], ref["force64"]) <= 1e-5
        assert np.abs(got["force"][:, 3] - ref["force64"][:, 3]).max() <= 1e-5 * max(np.abs(ref["force64"][:, 3]).max(), 1.0)
    patch, sim = marsmd.Patch(spec), orc.Sim(spec)
    patch.run(1)
    sim.run(1)
    got, ref = patch.copy_particles_to_host(), sim.copy_particles_to_host()
    assert np.array_equal(got["id"], ref["id"])
    d = np.abs(got["pos"][:, :3] - ref["pos"][:, :3])
    assert np.minimum(d, L - d).max() <= 1e-4


@pytest.mark.parametrize("limit", [1 << 15, 7 << 14])
def test_same_bits_on_both_sides_of_a_limit(cuda, limit):
    # `limit` beads around an empty sphere wider than the list cutoff; one more in its centre
    # has no neighbour, so every other bead's row and force are the same, summed by another
    # number of lanes
    L = (limit / 1.25e-4) ** (1.0 / 3.0)
    rs = np.random.default_rng(5)
    pos = rs.uniform(0.0, L, (limit + limit // 8, 3))
    pos = pos[np.linalg.norm(pos - L / 2, axis=1) > 40.0][:limit]
    assert len(pos) == limit
    out = []
    for extra in (0, 1):
        spec = configs.config0(n=8, L=L)
        spec.positions = np.vstack([pos, np.full((extra, 3), L / 2)]).astype(np.float32)
        spec.type_ids = np.zeros(limit + extra, np.int32)
        spec.params.energy_period = 1
        p = marsmd.Patch(spec)
        p.run(1)
        out.append(p.copy_particles_to_host()["force"][:limit])
    assert np.abs(out[0]).max() > 0
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
