"""Host threads that read one Patch or Batch at the same time: each gets whole records, the
same bits as a call by itself."""
import threading

import numpy as np
import pytest

import marsmd
from marsmd import configs
from marsmd.batch import Batch

pytestmark = pytest.mark.gpu

KEYS = ("pos", "mom", "force", "type", "id")


def _rows(records):
    records = records if isinstance(records, list) else [records]
    return [r[k] for r in records for k in KEYS]


@pytest.mark.parametrize("kind,n", [("patch", 501), ("patch", 300_007), ("batch", 90_000)])
def test_threads_read_whole_records(cuda, kind, n):
    if kind == "patch":
        spec = configs.config0(n=8, L=(n / 1e-4) ** (1.0 / 3.0))
        spec.positions = np.random.default_rng(n).uniform(0.0, spec.box.size[0], (n, 3)).astype(np.float32)
        spec.type_ids = np.zeros(n, np.int32)
        obj = marsmd.Patch(spec)
    else:
        obj = Batch(configs.config3(replicas=3, n_min=n // 3, n_max=n // 3, density=4e-4, seed=29))
    print("case:", kind, n, flush=True)
    want = _rows(obj.copy_particles_to_host())
    threads, wrong = 4, []
    start = threading.Barrier(threads)

    def read():
        start.wait()
        for _ in range(8):
            got = _rows(obj.copy_particles_to_host())
            if not all(np.array_equal(a, b) for a, b in zip(got, want)):
                wrong.append(1)

    team = [threading.Thread(target=read) for _ in range(threads)]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not wrong
