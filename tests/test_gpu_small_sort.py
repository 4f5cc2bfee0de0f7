"""The sort by one workgroup (up to 12288 keys) against numpy's stable sort, at the edges of
its batches, its waves' runs, its digits and its range; and the rebuilds' reductions, which
keep their accumulators from one call to the next."""

import numpy as np
import pytest

import marsmd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("key_bits", [1, 10, 11, 30, 32])
@pytest.mark.parametrize("n", [1, 15, 17, 64, 1023, 1025, 4097, 12287, 12288, 12289])
def test_small_sort_is_the_stable_sort_of_the_low_bits(cuda, n, key_bits):
    rs = np.random.default_rng(1000 * key_bits + n)
    keys = rs.integers(0, 2**32, size=n, dtype=np.uint64).astype(np.uint32)
    keys[::5] = keys[0]
    vals = rs.permutation(n).astype(np.uint32)
    kd, vd = (cuda.from_numpy(a.view(np.int32)).cuda() for a in (keys, vals))
    ko, vo = cuda.full((n + 1,), -7, dtype=cuda.int32, device="cuda"), cuda.full((n + 1,), -7, dtype=cuda.int32, device="cuda")
    nbytes = marsmd.lib().marsmd_radix_sort_scratch_bytes(n)
    scratch = cuda.empty(nbytes, dtype=cuda.uint8, device="cuda")
    marsmd._capi.call("marsmd_radix_sort_pairs", kd.data_ptr(), vd.data_ptr(), ko.data_ptr(), vo.data_ptr(), n,
                      key_bits, scratch.data_ptr(), nbytes, cuda.cuda.current_stream().cuda_stream)
    order = np.argsort(keys & np.uint32((1 << key_bits) - 1), kind="stable")
    assert np.array_equal(ko.cpu().numpy()[:n].view(np.uint32), keys[order])
    assert np.array_equal(vo.cpu().numpy()[:n].view(np.uint32), vals[order])
    assert int(ko[n]) == -7 and int(vo[n]) == -7
    assert np.array_equal(kd.cpu().numpy().view(np.uint32), keys)


@pytest.mark.parametrize("n", [2, 1024, 1025, 70_001])
def test_repeated_builds_and_displacements_start_from_zero(cuda, n):
    # a later call with smaller results must not see an earlier call's larger ones
    rs = np.random.default_rng(n)
    L = np.float32(4.0 * n ** (1 / 3) + 20.0)
    pos = cuda.zeros((n, 4), device="cuda")
    pos[:, :3] = cuda.from_numpy((rs.random((n, 3)) * 0.98 + 0.01).astype(np.float32) * L).cuda()
    pl = marsmd.ZOrderPairlist(n)
    pl.set_periodic_box(marsmd.PeriodicBox((float(L),) * 3))
    pairs = []
    for rc in (9.0, 5.0, 9.0):
        pl.build_pairlist(pos, n, rc)
        pairs.append(pl.get_num_pairs())
    assert pairs[0] == pairs[2] >= pairs[1]
    z = pl.get_sorter()
    z.update_positions_incremental(pos, n)
    for shift in (2.0, 0.5, 0.0):
        moved = pos.clone()
        moved[n // 2, 1] += shift
        want = abs(float(moved[n // 2, 1]) - float(pos[n // 2, 1]))
        assert pl.needs_update(moved, n, 2.0) == (want > 1.0)
        for d in (pl.last_max_displacement, z.compute_max_displacement(moved, n)):
            assert abs(d - want) <= 2.0**-22 * want  # a square and its root
