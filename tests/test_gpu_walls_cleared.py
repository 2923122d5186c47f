"""Walls that are cleared leave nothing behind: a wall added later starts at
time 0, however many one-launch steps ran with the old walls and without any
(dem_wall/src/lib.rs:766-815, the oscillation's phase)."""
import math
import sys

import numpy as np
import pytest

from mddem_amd import hip
from mddem_amd import workloads as W

pytestmark = pytest.mark.gpu

AMP, FREQ, Z0 = 2e-4, 2000.0, 0.001


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


@pytest.mark.parametrize("between", [0, 1, 2, 3, 6])
@pytest.mark.parametrize("first", [1, 20, 21])
def test_a_new_wall_starts_at_time_zero(first, between):
    w = W.dem_gas(n=100)
    s = hip.from_workload(w, hip.FP64, box_exit=False)
    s.add_wall((0, 0, 0.0005), (0, 0, 1))  # at rest
    s.run(first)
    s._c(s.L.mdd_clear_walls(s.h))
    s.run(between)
    s.add_wall((0, 0, Z0), (0, 0, 1))
    s.set_wall_motion(0, 2, (AMP, FREQ))
    steps = 3
    s.run(steps)
    z = Z0 + AMP * math.sin(2.0 * math.pi * FREQ * (steps * w.dt))
    got = s.walls()["point"][0]
    # time is summed step by step and the sine is the device's: a few ulp of Z0
    assert np.all(np.abs(got - [0.0, 0.0, z]) <= 8 * np.finfo(float).eps * Z0)
    # the oldest phase left over would show
    stale = Z0 + AMP * math.sin(2.0 * math.pi * FREQ * ((steps + 1) * w.dt))
    assert abs(stale - z) > 1e3 * np.finfo(float).eps * Z0
    s.close()
