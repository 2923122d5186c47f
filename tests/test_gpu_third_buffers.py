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


def test_a_long_run_makes_the_copy():
    # 50,000 spheres: 6.4 MB of second state after run(40), none after 40 x run(1)
    w = W.gas_system(50000, 0.2, 0.9, 0.4, seed=3)
    used = []
    for calls in ((40,), (1,) * 40):
        free = hip.device_memory(0)[0]
        s = hip.from_workload(w, hip.MIXED, box_exit=False)
        for k in calls:
            s.run(k)
        used.append(free - hip.device_memory(0)[0])
        s.close()
    assert used[0] - used[1] >= 4 * 32 * w.n - (2 << 20)


def _pair(w, prec, n, configure=lambda s: None):
    a, b = (hip.from_workload(w, prec, box_exit=False) for _ in range(2))
    configure(a)
    configure(b)
    a.run(n)
    for _ in range(n):
        b.run(1)
    return a, b


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("sign", [-1.0, 1.0])
def test_rebuilds_that_do_not_fit(sign, prec):
    # inward: rows outgrow their capacity; outward: the images near the faces do
    w = W.lj_fcc(ncell=5, rho=0.3, thermostat=False)
    L = w.hi - w.lo
    d = w.pos - (w.lo + 0.5 * L)
    d -= L * np.round(d / L)
    w.vel = sign * 1.2 * d / (0.5 * L)
    a, b = _pair(w, prec, 300)
    assert a.thermo()["rebuilds"] == b.thermo()["rebuilds"] > 3
    _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("steps", [400, 401])
def test_spheres_that_leave_through_fixed_faces(steps, prec):
    w = W.gas_system(700, 0.3, 0.9, 0.4, seed=3)
    w.vel = w.vel * 40.0
    w.omega = (W.Stream(6).uniform(3 * w.n).reshape(-1, 3) - 0.5) * 100.0
    w.periodic = (False, True, False)
    a, b = _pair(w, prec, steps)
    assert a.n == b.n and 100 < a.n < w.n - 20
    _same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("every", [2, 7])
def test_contact_virial_between_one_launch_steps(every, prec):
    w = W.dem_packed_bed(n=900, box=(0.02, 0.02, 0.2), vmax=0.02, seed=3)
    a, b = _pair(w, prec, 10 * every, lambda s: s.set_virial(every))
    _same(a, b)
    ta, tb = a.thermo(energy=True), b.thermo(energy=True)
    assert ta == tb and any(ta["virial"])
    a.close()
    b.close()
