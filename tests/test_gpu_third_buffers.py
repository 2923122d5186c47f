"""The second copy of the state that one-launch steps write: made when a run is
long enough, kept over uploads, remade when an upload outgrows it."""
import sys

import numpy as np
import pytest

from mddem_amd import hip
from mddem_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


def _workload(kind, big):
    # (at 20,000 particles the copy is past 2 MiB for spheres, at 42,592 for atoms)
    if kind == "lj":
        return W.lj_fcc(ncell=22 if big else 8, thermostat=False)
    w = W.gas_system(20000 if big else 700, 0.3, 0.9, 0.4, seed=3)
    w.vel = w.vel * 20.0
    w.omega = (W.Stream(6).uniform(3 * w.n).reshape(-1, 3) - 0.5) * 100.0
    return w


def _configure(s, w):
    s.set_box(w.lo, w.hi, w.periodic)
    s.upload(w.pos, w.vel, w.mass, w.cutoff_radius, radius=w.radius, omega=w.omega, tag=w.tag,
             atype=w.atype)


def _same(a, b):
    sa, sb = a.state(), b.state()
    for k in sb:
        assert np.array_equal(sa[k], sb[k]), k


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("kind", ["lj", "dem"])
@pytest.mark.parametrize("order", [(0, 1, 0), (1, 0, 1)])
@pytest.mark.parametrize("steps", [40, 41])
def test_uploads_of_other_sizes(kind, order, steps, prec):
    ws = [_workload(kind, k) for k in order]
    s = hip.from_workload(ws[0], prec, box_exit=False)
    s.run(steps)
    for w in ws[1:]:
        _configure(s, w)
        s.run(steps)
        ref = hip.from_workload(w, prec, box_exit=False)
        ref.run(steps)
        _same(s, ref)
        ref.close()
    s.close()


@pytest.mark.parametrize("kind", ["lj", "dem"])
def test_short_runs_and_a_long_one(kind):
    w = _workload(kind, 1)
    a = hip.from_workload(w, hip.MIXED, box_exit=False)
    b = hip.from_workload(w, hip.MIXED, box_exit=False)
    for k in (5, 10, 2, 20, 9, 30):
        a.run(k)
        for _ in range(k):
            b.run(1)
        _same(a, b)
    a.close()
    b.close()
