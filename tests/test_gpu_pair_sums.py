"""The pair forces of long lists (2^18 pairs and more are summed per workgroup in LDS) in the
orders a caller may bring, against the same pairs in short calls (which are not)."""
import numpy as np
import pytest

import marsmd
from marsmd import PeriodicBox
from oracle import pyoracle as orc
from tests.conftest import rel_force_error
from tests.test_gpu_analytical_terms import ANALYTIC, FORCE_TOL, _launch_inputs, analytic_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [(1 << 18) - 1, 1 << 18, (1 << 18) + 2047, 400_001])
@pytest.mark.parametrize("order", ["rows", "random", "one particle", "rows of a few"])
def test_long_lists_sum_to_their_parts(cuda, order, count):
    torch = cuda
    rs = np.random.default_rng(count)
    n, L = 20_011, 300.0
    pos = torch.zeros(n, 4, device="cuda")
    pos[:, :3] = torch.from_numpy(rs.random((n, 3), dtype=np.float32) * np.float32(L)).cuda()
    i = rs.integers(0, n, count)
    if order == "rows":
        i = np.sort(i)
    elif order == "one particle":
        i[:] = 7
    elif order == "rows of a few":
        i = np.sort(i) // 5 * 5
    pairs = torch.from_numpy(np.stack([i, (i + 1 + rs.integers(0, n - 1, count)) % n], axis=1).astype(np.int32)).cuda()
    cut, step = 60.0, 60.0 / 255
    tab = marsmd.TabulatedPotential(((np.arange(256) * step - 30.0) ** 2).astype(np.float32), 0.0, step)
    tables = marsmd.DeviceTables([tab])
    tags = torch.full((count,), marsmd._capi.PAIR_TERM_TABULATED, dtype=torch.int32, device="cuda")
    types = torch.zeros(n, dtype=torch.int32, device="cuda")

    def forces(chunk):
        fe = torch.zeros(n, 4, device="cuda")
        view = marsmd.particle_view(pos=pos, force_energy=fe, type_id=types)
        for a in range(0, count, chunk):
            part = pairs[a:a + chunk].contiguous()
            marsmd.launch_pairwise_nonbonded(part, view, tags[:len(part)], tables, PeriodicBox((L,) * 3), True,
                                             len(part), cut * cut)
        return fe.double()

    whole, parts = forces(count), forces(100_000)
    # either order rounds each of a particle's k additions by at most 2^-24 of the sum of its
    # terms' magnitudes (the table's slope and value at the pair's distance, one bin off at most)
    d = pos[pairs[:, 0].long(), :3].double() - pos[pairs[:, 1].long(), :3].double()
    d = (d - L * torch.round(d / L)).norm(dim=1)
    near = d <= cut + 1e-3
    assert int(near.sum()) > 1000
    mag = torch.stack([(2.0 * (d - 30.0).abs() + 2.0 * step) * near, ((d.clamp(max=cut) - 30.0) ** 2 + 30.0) * near / 2,
                       near.double()], dim=1)
    total = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
    for end in (0, 1):
        total.index_add_(0, pairs[:, end].long(), mag)
    bound = 2.0 * 2.0**-24 * total[:, 2:] * total[:, [0, 0, 0, 1]]
    assert bool(((whole - parts).abs() <= bound).all())
    assert float(whole[:, 3].sum()) > 0.0


@pytest.mark.parametrize("terms", [ANALYTIC, ANALYTIC | marsmd._capi.PAIR_TERM_TABULATED])
def test_long_lists_with_analytical_terms_match_the_oracle(cuda, terms):
    spec = analytic_spec(n=3000, L=110.0, seed=9)
    pos, pairs, tags, pd, td, tag_d = _launch_inputs(cuda, spec)
    assert len(pairs) >= 1 << 18
    fe = cuda.zeros((len(pos), 4), dtype=cuda.float32, device="cuda")
    pos_d, cut2 = cuda.from_numpy(pos).cuda(), spec.params.cutoff ** 2
    if terms == ANALYTIC:
        marsmd.launch_analytical_pair_nonbonded(pd, pos_d, fe, td, tag_d, spec.types, spec.box, terms, True,
                                                len(pairs), cut2, params=spec.pair_params)
    else:
        view = marsmd.particle_view(pos=pos_d, force_energy=fe, type_id=td)
        marsmd.launch_pairwise_nonbonded(pd, view, tag_d, marsmd.DeviceTables(spec.nb_tables), spec.box, True,
                                         len(pairs), cut2, terms, types=spec.types, params=spec.pair_params)
    ref = orc.pair_forces(pairs, pos, spec.type_ids, tags, spec.nb_tables, spec.box, cut2, mode=1,
                          enabled_terms=terms, particle_types=spec.types, pair_params=spec.pair_params)
    g = fe.cpu().numpy()
    assert rel_force_error(g, ref) <= FORCE_TOL
    assert abs(g[:, 3].sum() - ref[:, 3].sum()) <= 1e-5 * np.abs(ref[:, 3]).sum()
