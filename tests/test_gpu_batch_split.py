"""The batch step at the edges of its row split (8 lanes a row up to 2^15 slots, 4 up to
7 2^14, then 1): every replica against its own Patch."""
import dataclasses

import numpy as np
import pytest

import marsmd
from marsmd import configs
from marsmd.batch import Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("integrator", [marsmd._capi.INTEGRATOR_BROWNIAN, marsmd._capi.INTEGRATOR_LANGEVIN])
@pytest.mark.parametrize("sizes", [[300, 500, 1000], [8192] * 3 + [8191], [8192] * 4, [8192] * 3 + [8193],
                                   [28672] * 4, [28672] * 3 + [28673]])
def test_batch_step_matches_single_patches(cuda, sizes, integrator):
    specs = []
    for r, n in enumerate(sizes):
        s = configs.config3(replicas=1, n_min=n, n_max=n, density=4e-4, seed=29)[0]
        assert s.n == n
        # (short Langevin steps: a bead of the random start deep in another's core would
        # carry one rounding of its force away)
        dt = s.params.timestep * (1.0 if integrator == marsmd._capi.INTEGRATOR_BROWNIAN else 1e-2)
        specs.append(dataclasses.replace(s, patch_id=r, params=dataclasses.replace(
            s.params, integrator=integrator, timestep=dt, energy_period=4)))
    b = Batch(specs)
    b.run(9)
    got = b.copy_particles_to_host()
    for r, s in enumerate(specs):
        p = marsmd.Patch(s)
        p.run(9)
        h = p.copy_particles_to_host()
        assert np.array_equal(got[r]["id"], h["id"])
        d = np.abs(got[r]["pos"][:, :3] - h["pos"][:, :3])
        assert np.minimum(d, s.box.size[0] - d).max() < 1e-3, f"replica {r} of {len(sizes)}"
        # the row order, and with it the sums, may differ: 2^-24 of the terms a few hundred times
        scale = np.abs(h["force"]).max() + 1.0
        assert np.abs(got[r]["force"] - h["force"]).max() < 2e-4 * scale
