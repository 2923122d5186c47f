"""Admission's estimate of a job's device memory covers what its context
allocates, a run and a download included."""
import sys

import pytest

from mddem_amd import hip, serve

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("kind", ["dem", "lj", "lj_nve"])
def test_estimate_covers_the_allocations(kind, prec):
    # the largest sizes of the job stream, where the fixed part counts least
    model = kind.split("_")[0]
    job = serve.Job(0, model, dict(dem=200_000, lj=500_000)[model], 100, 0.0,
                    dict(seed=11, rho=0.9, temperature=1.2))
    w = job.workload = serve.build_workload(job)
    if kind == "lj_nve":
        w.nose_hoover = None
    hip.System(hip.MODEL_LJ).close()  # what a process allocates once
    free = hip.device_memory(0)[0]
    s = hip.from_workload(w, prec, box_exit=False)
    s.run(job.steps)
    s.state()
    used = free - hip.device_memory(0)[0]
    s.close()
    assert used <= serve.FOOTPRINT_PER_PARTICLE[model] * w.n
