"""The cell configuration that the getters report is the one in use: the default stands for
the library's own choice, and setting what a getter reported brings the same rows (the
order of the pairs) back."""
import dataclasses

import numpy as np
import pytest

import marsmd
from marsmd import configs
from marsmd.batch import Batch
from marsmd.core import PeriodicBox

pytestmark = pytest.mark.gpu


def _patch_rows(spec, cells=()):
    p = marsmd.Patch(spec)
    for c in cells:
        p.set_cells(*c)
        assert p.get_cells() == c
    p.run(1)
    return p.get_pairlist().get_neighbor_pairs().cpu().numpy()


@pytest.mark.parametrize("periodic", [(True, True, True), (False, True, True), (False, False, False)])
def test_patch_default_cells_come_back(cuda, periodic):
    spec = configs.config0(n=6000, L=300.0, seed=3)
    spec.box = PeriodicBox((300.0,) * 3, periodic=periodic)
    default = marsmd.Patch(spec).get_cells()
    own, tuned = _patch_rows(spec), _patch_rows(spec, [(8, 3)])
    assert len(own) == len(tuned) and not np.array_equal(own, tuned)
    assert np.array_equal(_patch_rows(spec, [(8, 3), default]), own)
    assert np.array_equal(_patch_rows(spec, [default]), own)


def _batch_rows(specs, cells=()):
    b = Batch(specs)
    for c in cells:
        b.set_cells(c)
        assert b.get_cells() == c
    b.run(1)
    return np.concatenate([b.get_neighbor_pairs(r) for r in range(len(specs))])


def test_batch_default_cells_come_back(cuda):
    specs = configs.config3(replicas=4, n_min=2500, n_max=7000, density=4e-4, seed=17)
    default = Batch(specs).get_cells()
    other = {b: (8, 3) for b in default}
    own, tuned = _batch_rows(specs), _batch_rows(specs, [other])
    assert len(own) == len(tuned) and not np.array_equal(own, tuned)
    assert np.array_equal(_batch_rows(specs, [other, default]), own)
    assert np.array_equal(_batch_rows(specs, [default]), own)


def test_tuned_cells_give_the_tuned_rows(cuda):
    # dt = 0: every build sees the same positions
    spec = configs.config0(n=6000, L=300.0, seed=3)
    spec.box = PeriodicBox((300.0,) * 3, periodic=(False, True, True))
    spec.params = dataclasses.replace(spec.params, timestep=0.0, rebuild_period=5, reorder_period=1000)
    p = marsmd.Patch(spec)
    choice = p.autotune_cells(12)
    print("case: tuned cells", choice, flush=True)
    rows = p.get_pairlist().get_neighbor_pairs().cpu().numpy()
    assert np.array_equal(_patch_rows(spec, [(choice["home_target"], choice["fine_offset"])]), rows)
    specs = configs.config3(replicas=4, n_min=2500, n_max=7000, density=4e-4, seed=17)
    for s in specs:
        s.params = dataclasses.replace(s.params, timestep=0.0, rebuild_period=5, reorder_period=1000)
    b = Batch(specs)
    cells = b.autotune_cells(12, cache=False)["cells"]
    print("case: tuned cells", cells, flush=True)
    b.run(5, first_step=20)  # past a build with the choice
    rows = np.concatenate([b.get_neighbor_pairs(r) for r in range(len(specs))])
    assert np.array_equal(_batch_rows(specs, [cells]), rows)
