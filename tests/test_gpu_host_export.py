"""Particle records to host arrays, in pieces: sizes at the edges of a piece (16384 particles)
and of the staging memory (16 pieces), against the particles that went in."""
import dataclasses

import numpy as np
import pytest

import marsmd
from marsmd import PeriodicBox, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 501, 16_383, 16_384, 16_385, 49_153, 262_144, 262_145, 300_007])
def test_records_come_back_as_they_went_in(cuda, n):
    rs = np.random.default_rng(n)
    base = configs.config3(replicas=1, n_min=300, n_max=400, density=4e-4, seed=3)[0]
    spec = dataclasses.replace(base, box=PeriodicBox((400.0,) * 3),
                               positions=rs.random((n, 3), dtype=np.float32) * np.float32(400.0),
                               momenta=rs.standard_normal((n, 3)).astype(np.float32),
                               type_ids=rs.integers(0, len(base.types), n).astype(np.int32))
    patch = marsmd.Patch(spec)
    for _ in range(2):  # the staging memory is kept
        h = patch.copy_particles_to_host()
        assert np.array_equal(h["pos"], spec.pos4())
        assert np.array_equal(h["mom"][:, :3], spec.momenta)
        assert not h["force"].any()
        assert np.array_equal(h["type"], spec.type_ids)
        assert np.array_equal(h["id"], np.arange(n, dtype=np.int32))
    # the first particles only, into some of the arrays
    m = (n + 1) // 2
    pos, ids = np.full((n, 4), -1.0, np.float32), np.full(n, -1, np.int32)
    marsmd._capi.call("marsmd_patch_copy_particles_to_host", patch._h, pos.ctypes.data, None, None, None,
                      ids.ctypes.data, m)
    assert np.array_equal(pos[:m], spec.pos4()[:m]) and (pos[m:] == -1.0).all()
    assert np.array_equal(ids[:m], np.arange(m)) and (ids[m:] == -1).all()
