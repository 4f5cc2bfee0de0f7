"""New particles uploaded to a batch that has run: the runs that follow are those of a batch
made with these particles."""
import numpy as np
import pytest

from marsmd import _capi as api
from marsmd import configs
from marsmd.batch import Batch
from oracle import pyoracle as orc
from tests.conftest import sorted_pairs

pytestmark = pytest.mark.gpu


def _specs():
    return configs.config3(replicas=4, n_min=300, n_max=1500, density=4e-4, seed=17)


@pytest.mark.parametrize("integrator", [api.INTEGRATOR_BROWNIAN, api.INTEGRATOR_LANGEVIN])
@pytest.mark.parametrize("steps", [1, 25, 65])  # before the second build, past it, past later ones
def test_upload_to_a_batch_that_has_run(cuda, steps, integrator):
    specs, again = _specs(), _specs()
    params = configs.RunParams(cutoff=30.0, pairlist_cutoff=35.0, rebuild_period=10, reorder_period=20,
                               timestep=1e-4 if integrator == api.INTEGRATOR_BROWNIAN else 2e-5, kT=configs.KT,
                               integrator=integrator)
    for r, s in enumerate(again):
        s.positions = configs.uniform_positions(s.n, s.box.size[0], 1000 * steps + r)
    print("case:", steps, integrator, flush=True)
    b = Batch(specs)
    b.run(steps, params=params)
    pos = np.concatenate([s.pos4() for s in again])
    types = np.concatenate([np.asarray(s.type_ids, np.int32) for s in again])
    api.call("marsmd_batch_copy_particles_from_host", b._h, pos.ctypes.data, None, types.ctypes.data, b.total)
    for s in again:
        s.momenta = None
    fresh = Batch(again)
    first = 0
    for chunk in (1, 30):
        b.run(chunk, first_step=first, params=params)
        fresh.run(chunk, first_step=first, params=params)
        first += chunk
        if chunk == 1:
            for r, s in enumerate(again):
                ref = orc.build_pairlist(s.pos4(), s.box, params.pairlist_cutoff)["pairs"].astype(np.int64)
                assert np.array_equal(sorted_pairs(b.get_neighbor_pairs(r)), ref), f"replica {r}"
        got, want = b.copy_particles_to_host(), fresh.copy_particles_to_host()
        for r in range(len(again)):
            for k in ("pos", "mom", "force", "id"):
                assert np.array_equal(got[r][k], want[r][k]), f"replica {r}: {k} after {first} steps"
