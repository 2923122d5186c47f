"""Either side of the lines up to which steps go in one launch: run(N) is
N x run(1) (separate passes) bit for bit."""
import sys

import numpy as np
import pytest

from mddem_amd import hip
from mddem_amd import workloads as W

pytestmark = pytest.mark.gpu

STEPS = 35


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


def _gas(n, phi):
    w = W.gas_system(n, phi, 0.9, 0.4, seed=5)
    w.vel = w.vel * 20.0
    w.omega = (W.Stream(6).uniform(3 * n).reshape(-1, 3) - 0.5) * 100.0
    return w


def _runs_alike(w, prec, configure):
    a, b = (hip.from_workload(w, prec, box_exit=False) for _ in range(2))
    configure(a)
    configure(b)
    a.run(STEPS)
    for _ in range(STEPS):
        b.run(1)
    sa, sb = a.state(), b.state()
    for k in sb:
        assert np.array_equal(sa[k], sb[k]), k
    for x, y in zip(a.forces(), b.forces()):
        assert np.array_equal(x, y)
    a.close()
    b.close()


def _cloud_on_a_floor(n):
    # spheres moving between two planes under gravity
    w = W.dem_settling(n=n, box=(0.06, 0.06, 0.3))
    w.vel = (W.Stream(9).uniform(3 * n).reshape(-1, 3) - 0.5) * 4.0
    w.omega = (W.Stream(6).uniform(3 * n).reshape(-1, 3) - 0.5) * 100.0
    return w


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("split", [-1, 1])
@pytest.mark.parametrize("n", [1, 257, 3001])
def test_split_by_row_length(n, split, prec):
    def configure(s):
        s.set_force_lanes(0)
        s.set_dem_split(split)

    _runs_alike(_cloud_on_a_floor(n), prec, configure)


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("lanes,n", [(3, 49999), (3, 50000), (2, 199999), (2, 200000)])
def test_lanes(lanes, n, prec):
    _runs_alike(_gas(n, 0.3), prec, lambda s: s.set_force_lanes(lanes))
