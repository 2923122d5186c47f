"""A run that the overlap limit stops (dem_granular/src/contact.rs:103-615,
more than 500 overlaps past 10% in one step) leaves the particles where the
step's first half put them, every particle of the same step: run(N) with one
launch per step the same as N x run(1) with separate passes, bit for bit."""
import sys

import numpy as np
import pytest

from mddem_amd import hip
from mddem_amd import workloads as W

pytestmark = pytest.mark.gpu

PAIRS = 650


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


def _colliding_pairs():
    # pairs on a grid of 6 radii, 1.15 diameters apart, closing by 0.06
    # diameters a step: no contact gets past 0.91 before the fifth step, where
    # all are at 0.85. The spheres spin.
    w = W.dem_gas(n=2 * PAIRS, box=0.09)
    r = 1e-3
    g = np.stack(np.meshgrid(*[np.arange(9)] * 3, indexing="ij"), -1).reshape(-1, 3)[:PAIRS]
    mid = (g + 0.5) * 6.0 * r
    d = np.array([1.15 * r, 0.0, 0.0])
    w.hi = w.lo + 9 * 6.0 * r
    w.pos = np.concatenate([mid - d, mid + d])
    v = np.array([0.06 * r / w.dt, 0.0, 0.0])
    w.vel = np.concatenate([np.tile(v, (PAIRS, 1)), np.tile(-v, (PAIRS, 1))])
    w.omega = (W.Stream(8).uniform(6 * PAIRS).reshape(-1, 3) - 0.5) * 400.0
    assert np.all(w.radius == r)
    return w


def _system(w, prec, shape):
    s = hip.from_workload(w, prec, box_exit=False)
    if shape == "cohesive":
        s.set_material_extras(cohesion_energy=[5e3])
    elif shape != "auto":
        s.set_force_lanes(int(shape[0]))
        s.set_dem_wave(shape.endswith("queue"))
        s.set_dem_split(1 if shape.endswith("split") else 0)
    return s


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("skin", [1.1, 1.8])  # with rebuilds on the way, and without
@pytest.mark.parametrize("shape", ["auto", "0", "0 queue", "0 split", "2", "cohesive"])
def test_the_stopped_state_is_of_one_step(shape, skin, prec):
    w = _colliding_pairs()
    w.skin_fraction = skin
    a = _system(w, prec, shape)
    with pytest.raises(hip.MddError) as ea:
        a.run(12)
    b = _system(w, prec, shape)
    done = 0
    with pytest.raises(hip.MddError) as eb:
        for _ in range(12):
            b.run(1)
            done += 1
    assert ea.value.code == eb.value.code and "overlaps" in str(ea.value)
    assert done == 4
    sa, sb = a.state(), b.state()
    for k in sb:
        assert np.array_equal(sa[k], sb[k]), k
    a.close()
    b.close()
