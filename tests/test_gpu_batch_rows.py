"""A replica's rows, and with them the bits of its forces and trajectory, do not depend on
the replicas beside it: the same alone, in a batch of several, and as a Patch."""
import dataclasses

import numpy as np
import pytest

import marsmd
from marsmd import _capi as api
from marsmd import configs
from marsmd.batch import Batch

pytestmark = pytest.mark.gpu

KEYS = ("pos", "mom", "force", "id")


# sizes at the walk's level changes; dense ones in boxes that the cutoff spans on every axis
@pytest.mark.parametrize("density", [1e-4, 8e-4])
@pytest.mark.parametrize("sizes", [[60, 191, 192, 500], [1474, 1024, 8192, 300], [4000, 12_287, 12_288, 900],
                                   [16_384, 16_385, 30_011]])
@pytest.mark.parametrize("integrator", [api.INTEGRATOR_BROWNIAN, api.INTEGRATOR_LANGEVIN])
def test_a_replica_keeps_its_bits(cuda, sizes, density, integrator):
    specs = []
    for r, n in enumerate(sizes):
        s = configs.config3(replicas=1, n_min=n, n_max=n, density=density, seed=29)[0]
        assert s.n == n
        specs.append(dataclasses.replace(s, patch_id=r, params=dataclasses.replace(
            s.params, integrator=integrator, timestep=s.params.timestep / 100.0, rebuild_period=5, energy_period=4)))
    steps = 12
    b = Batch(specs)
    b.run(steps)
    together = b.copy_particles_to_host()
    for r, s in enumerate(specs):
        print("case:", density, integrator, s.n, flush=True)
        one = Batch([s])
        one.run(steps)
        alone = one.copy_particles_to_host()[0]
        p = marsmd.Patch(s)
        p.run(steps)
        patch = p.copy_particles_to_host()
        assert np.abs(alone["force"]).max() > 0
        for k in KEYS:
            assert np.array_equal(together[r][k], alone[k]), f"{k} of {s.n} beads in a batch"
            assert np.array_equal(together[r][k], patch[k]), f"{k} of {s.n} beads against a Patch"


@pytest.mark.parametrize("replicas", [3, 40, 200])
@pytest.mark.parametrize("n,density", [(500, 1e-4), (300, 1e-4), (1600, 8e-4)])
def test_a_replica_keeps_its_bits_in_a_crowd(cuda, n, density, replicas):
    # more replicas, coarser cells each: whole boxes, then a list for each home cell
    base = configs.config3(replicas=1, n_min=n, n_max=n, density=density, seed=29)[0]
    specs = []
    for r in range(replicas):
        s = dataclasses.replace(base, patch_id=r, params=dataclasses.replace(
            base.params, timestep=base.params.timestep / 100.0, rebuild_period=5))
        s.positions = configs.uniform_positions(n, base.box.size[0], 100 + r)
        specs.append(s)
    print("case:", n, density, replicas, flush=True)
    b = Batch(specs)
    b.run(7)
    together = b.copy_particles_to_host()
    for r in (0, replicas - 1):
        p = marsmd.Patch(specs[r])
        p.run(7)
        patch = p.copy_particles_to_host()
        for k in KEYS:
            assert np.array_equal(together[r][k], patch[k]), f"{k} of replica {r}"
