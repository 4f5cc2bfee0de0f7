"""The step with one lane to a row, which serves systems above 7 2^14 slots with short rows:
the bits of the step that deals a row to several lanes (one bead less), the oracle's forces
with bonded terms, and the same bits with pruned rows and with the grid force in a kernel of
its own."""
import re

import numpy as np
import pytest

import marsmd
from marsmd import _capi as api
from marsmd import configs
from oracle import pyoracle as orc
from tests.conftest import rel_force_error
from tests.test_gpu_analytical_terms import analytic_spec

pytestmark = pytest.mark.gpu

LIMIT = 7 << 14  # slots up to which four lanes share a row


def _langevin_cubic(n, L):
    return configs.config2(n=n, L=L, grid_n=64)


def _brownian_linear(n, L):
    spec = _langevin_cubic(n, L)
    spec.params.integrator = api.INTEGRATOR_BROWNIAN
    spec.params.interpolation = api.INTERP_LINEAR
    return spec


def _langevin_analytic(n, L):
    spec = analytic_spec(n=n, L=L)
    spec.types = [type(t)(**{**t.__dict__, "trans_damping": (1000.0,) * 3, "mass": 100.0}) for t in spec.types]
    spec.params.integrator = api.INTEGRATOR_LANGEVIN
    spec.params.timestep = 1e-6
    return spec


CASES = {"langevin_cubic": _langevin_cubic, "brownian_linear": _brownian_linear, "brownian_table": configs.config0,
         "brownian_analytic": analytic_spec, "langevin_analytic": _langevin_analytic}


def _state(p):
    g = p.copy_particles_to_host()
    return {k: g[k].view(np.uint32) for k in ("pos", "mom", "force", "id")}


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("energy", [False, True])
@pytest.mark.parametrize("case", list(CASES))
def test_bits_of_the_split_rows(cuda, case, energy, given):
    # LIMIT beads around an empty sphere wider than the list cutoff, one more in its centre
    # without neighbours: every other bead's row and force are the same
    L = (LIMIT / 1.25e-4) ** (1.0 / 3.0)
    rs = np.random.default_rng(5)
    pos = rs.uniform(0.0, L, (LIMIT + LIMIT // 8, 3))
    pos = pos[np.linalg.norm(pos - L / 2, axis=1) > 40.0][:LIMIT]
    assert len(pos) == LIMIT
    print("case:", case, energy, given, flush=True)
    out = []
    for extra in (0, 1):
        spec = CASES[case](n=9, L=L)
        n = LIMIT + extra
        spec.positions = np.vstack([pos, np.full((extra, 3), L / 2)]).astype(np.float32)
        spec.type_ids = (np.arange(n) % len(spec.types)).astype(np.int32)
        if spec.momenta is not None:
            spec.momenta = np.random.default_rng(6).standard_normal((n, 3)).astype(np.float32)
        spec.params.energy_period = 1 if energy else 0
        p = marsmd.Patch(spec)
        p.set_launch(0, given)
        p.run(1)
        out.append({k: v[:LIMIT] for k, v in _state(p).items()})
    assert np.abs(out[0]["force"].view(np.float32)).max() > 0
    for k in out[0]:
        assert np.array_equal(out[0][k], out[1][k]), k


@pytest.mark.parametrize("case", ["langevin_cubic", "brownian_linear", "brownian_analytic"])
def test_options_keep_the_bits(cuda, case):
    n = LIMIT + 77
    spec = CASES[case](n=n, L=(n / 1.25e-4) ** (1.0 / 3.0))
    spec.params.energy_period = 7
    spec.params.reorder_period = 20
    if spec.params.integrator == api.INTEGRATOR_LANGEVIN:
        spec.params.timestep /= 50.0  # displacements inside the skin: the adaptive margin prunes

    def run(mode, margin, given):
        p = marsmd.Patch(spec)
        p.set_pruning(mode, margin)
        p.set_launch(0, given)
        out = []
        for first, steps in ((0, 13), (13, 9), (22, 23)):
            p.run(steps, first_step=first)
            out.append(_state(p))
        return out

    want = run(0, -1.0, False)
    for mode, margin, given in [(1, -1.0, False), (2, -1.0, False), (2, 1e-4, False), (2, 0.05, True),
                                (3, -1.0, False), (0, -1.0, True)]:
        print("case:", case, mode, margin, given, flush=True)
        for k, (a, b) in enumerate(zip(run(mode, margin, given), want)):
            for name in a:
                assert np.array_equal(a[name], b[name]), f"{name} after run {k}"


def test_bonded_terms_match_the_oracle(cuda):
    # chains of 225 beads with short rows (a cutoff of a few bonds)
    spec = configs.config1(chains=512, beads=225, L=1000.0, dihedrals=True, restraints=True)
    assert spec.n > LIMIT
    spec.params.cutoff, spec.params.pairlist_cutoff, spec.params.energy_period = 13.0, 15.0, 1
    patch, sim = marsmd.Patch(spec), orc.Sim(spec)
    patch.run(1)
    sim.run(1)
    got, ref = patch.copy_particles_to_host(), sim.copy_particles_to_host()
    stats = patch.get_pairlist().get_statistics()
    assert 2 * patch.get_pairlist().get_num_pairs() < 48 * spec.n, stats  # short rows: one lane each
    assert np.array_equal(got["id"], ref["id"])
    assert rel_force_error(got["force"], ref["force64"]) <= 1e-5
    d = np.abs(got["pos"][:, :3] - ref["pos"][:, :3])
    assert np.minimum(d, 1000.0 - d).max() <= 1e-3


@pytest.mark.parametrize("n,lanes_kernel", [(20_000, "k_step_split<"), (LIMIT, "k_step_split<"), (LIMIT + 1, "k_step<")])
@pytest.mark.parametrize("given", [False, True])
def test_the_kernels_that_run(cuda, n, lanes_kernel, given):
    # the launch option decides where the grid force comes from, whatever deals the rows
    from torch.profiler import ProfilerActivity, profile

    L = (n / 1.25e-4) ** (1.0 / 3.0)
    spec = _brownian_linear(9, L)
    spec.positions = np.random.default_rng(8).uniform(0.0, L, (n, 3)).astype(np.float32)
    spec.type_ids = (np.arange(n) % 3).astype(np.int32)
    spec.momenta = None
    p = marsmd.Patch(spec)
    p.set_launch(0, given)
    p.run(1)
    cuda.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        p.run(3, first_step=1)
        cuda.cuda.synchronize()
    names = [e.name for e in prof.events()]
    if not any("mmd::" in x for x in names):
        pytest.skip("the profiler records no kernels here")
    steps = [x for x in names if "k_step<" in x or "k_step_split<" in x]
    assert len(steps) == 3 and all(lanes_kernel in x for x in steps), names
    assert sum("k_pmf_force" in x for x in names) == (3 if given else 0), names
    # the fourth template argument: sampled linearly here (1) or given (3)
    assert all(re.search(r"<[^,]*, [^,]*, [^,]*, (\d)", x).group(1) == ("3" if given else "1") for x in steps), steps


@pytest.mark.parametrize("energy", [0, 2])
@pytest.mark.parametrize("case", ["brownian_table", "brownian_analytic", "langevin_analytic"])
def test_batch_replicas_have_the_bits_of_patches(cuda, case, energy):
    # 5 replicas together take one lane a row, each as a Patch four
    from marsmd.batch import Batch

    specs = []
    for r, n in enumerate([24_000, 23_999, 20_011, 25_000, 24_001]):
        spec = CASES[case](n=n, L=(n / 1.25e-4) ** (1.0 / 3.0))
        spec.patch_id, spec.params.energy_period, spec.params.rebuild_period = r, energy, 3
        spec.params.timestep /= 50.0
        specs.append(spec)
    assert sum(s.n for s in specs) > LIMIT
    print("case:", case, energy, flush=True)
    b = Batch(specs)
    b.run(6)
    for r, (spec, got) in enumerate(zip(specs, b.copy_particles_to_host())):
        p = marsmd.Patch(spec)
        p.run(6)
        for k, want in _state(p).items():
            assert np.array_equal(got[k].view(np.uint32), want), f"{k} of replica {r}"
