"""A Patch's pairlist in a caller's hands: exclusion rows that are not symmetric or name
particles outside the build, and fewer particles than the Patch's own rows name, against
the oracle's pairlist (bit for bit the same set)."""
import numpy as np
import pytest

import marsmd
from marsmd import configs
from marsmd.core import ExclusionCSR
from oracle import pyoracle as orc
from tests.conftest import sorted_pairs

pytestmark = pytest.mark.gpu


def _patch():
    spec = configs.config1(chains=12, beads=60, L=120.0, seed=5)
    patch = marsmd.Patch(spec)
    patch.run(1)
    return spec, patch


def _pairs(cuda, pl, pos, rc):
    pl.build_pairlist(cuda.from_numpy(pos).cuda(), len(pos), rc)
    return sorted_pairs(pl.get_neighbor_pairs().cpu().numpy())


@pytest.mark.parametrize("beyond", [False, True])
def test_asymmetric_rows_on_a_patch_pairlist(cuda, beyond):
    spec, patch = _patch()
    n, rc, pos = spec.n, spec.params.pairlist_cutoff, spec.pos4()
    near = orc.build_pairlist(pos, spec.box, rc)["pairs"]
    rs = np.random.default_rng(3)
    off, exc, ne = marsmd.exclusion_csr_from_pairs(near[rs.permutation(len(near))[:3000]])
    rows = [exc[off[i]:off[i + 1]][::2] for i in range(ne)]  # every other entry of every row
    if beyond:  # and particles far outside the build, which exclude nothing
        rows = [np.concatenate([[n + 7, 1 << 30], r, [2**31 - 1]]) for r in rows]
    off = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    exc = np.concatenate(rows).astype(np.int32)
    pl = patch.get_pairlist()
    print("case: rows beyond the build", beyond, flush=True)
    pl.set_exclusions(ExclusionCSR(offsets=cuda.from_numpy(off).cuda(), excluded=cuda.from_numpy(exc).cuda(),
                                   num_particles=ne))
    want = orc.build_pairlist(pos, spec.box, rc, offsets=off, excluded=exc, num_excl=ne)["pairs"].astype(np.int64)
    assert np.array_equal(_pairs(cuda, pl, pos, rc), want)


def test_fewer_particles_than_the_patch_rows_name(cuda):
    # 331 beads: the last chain is cut, so its rows name beads that are not in the call
    spec, patch = _patch()
    rc, pos = spec.params.pairlist_cutoff, spec.pos4()[:331]
    off, exc, ne = marsmd.exclusion_csr_from_pairs(spec.exclusions)
    want = orc.build_pairlist(pos, spec.box, rc, offsets=off, excluded=exc, num_excl=ne)["pairs"].astype(np.int64)
    assert np.array_equal(_pairs(cuda, patch.get_pairlist(), pos, rc), want)
