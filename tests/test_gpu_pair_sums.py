"""The pair forces of long lists (2^18 pairs and more are summed per workgroup in LDS) in the
orders a caller may bring, against the same pairs in short calls (which are not)."""
import numpy as np
import pytest

import marsmd
from marsmd import PeriodicBox

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
