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
