"""The pair passes read a row's first entries before they know its length:
rows shorter than that, empty ones, the last particles of a launch and a list
whose rows hold fewer entries than are read ahead. Forces against the oracle;
the layouts of the one row list against each other."""
import sys

import numpy as np
import pytest

from mddem_amd import hip
from mddem_amd import workloads as W
from tests.helpers import oracle_from_workload, rel_err
from tests.test_gpu_parity import FP64_TOL, MIXED_TOL, _oracle_rebuild, by_tag

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


def _chain(n, kind):
    """n particles in a row, each within reach of the next, except that every
    seventh gap is too wide: rows of 0, 1 and 2 entries."""
    w = W.lj_fcc(ncell=3) if kind == "lj" else W.dem_gas(n=64, box=0.025)
    r = 0.5 if kind == "lj" else 1e-3
    gap = 2.0 * r * (1.0 if kind == "lj" else 0.999)
    x = np.cumsum(np.where(np.arange(n) % 7 == 3, 3.5 * gap, gap))
    L = np.array([x[-1] + 30.0 * r, 30.0 * r, 30.0 * r])
    w.lo, w.hi = np.zeros(3), L
    w.pos = np.column_stack([x, np.full(n, 15.0 * r), np.full(n, 15.0 * r)])
    w.vel = np.zeros((n, 3))
    w.mass = np.full(n, float(w.mass[0]))
    w.cutoff_radius = np.full(n, r)
    w.skin_fraction = 1.02
    w.atype = None
    if kind != "lj":
        w.radius = np.full(n, r)
        if w.omega is not None:
            w.omega = np.zeros((n, 3))
    return w


@pytest.mark.parametrize("lanes", [None, 0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 2, 63, 130, 257])
@pytest.mark.parametrize("kind", ["lj", "dem"])
def test_short_rows(kind, n, lanes):
    w = _chain(n, kind)
    o = oracle_from_workload(w)
    _oracle_rebuild(o)
    o.zero_all_forces()
    (o.lj_force if kind == "lj" else o.hertz_mindlin_contact_force)()
    o.reverse_send_force()
    ref = o.atoms()
    for prec, tol in ((hip.FP64, FP64_TOL), (hip.MIXED, MIXED_TOL)):
        s = hip.from_workload(w, prec)
        if lanes is not None:
            s.set_force_lanes(lanes)
        s.bin_neighbor_list()
        (s.lj_force if kind == "lj" else s.hertz_mindlin_contact_force)()
        f = by_tag(s.state()["tag"], s.forces()[0])
        g = by_tag(ref["tag"], ref["force"])
        assert np.any(g != 0.0) == (n > 1)
        assert rel_err(f, g) < tol
        s.close()
