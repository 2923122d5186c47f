"""Rows of a batch by wavefronts that take a cell and by lanes that take a
member are the same: the same pairs, and runs that agree bit for bit, which
the lanes take by themselves where the batch has fewer spheres than cells."""
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


def _systems(kind):
    # systems of uneven size, density and box; "poly": of unequal spheres, where
    # each pair has a cutoff of its own
    ns = dict(one=[1], small=[1, 2, 65, 200], uneven=[200, 3001, 17, 900], poly=[300, 64, 700])[kind]
    out = []
    for k, n in enumerate(ns):
        w = W.gas_system(n, (0.05, 0.3, 0.15, 0.25)[k % 4], 0.9, 0.4, seed=40 + k)
        if kind == "poly":
            w.radius = w.radius * (0.8 + 0.2 * W.Stream(k).uniform(n))
            w.cutoff_radius = w.radius.copy()
        w.vel = w.vel * 20.0
        out.append(w)
    return out


def _run(systems, prec, mode, bins):
    s = hip.System(hip.MODEL_DEM, prec)
    s.set_neighbor(1.1, bins * 2.2e-3, 0, True, 1000, True)
    s.set_dt(systems[0].dt)
    s.set_build_kernel(mode)
    for w in systems:
        m = w.materials
        s.add_system(w.lo, w.hi, m["youngs"][0], m["poisson"][0], m["restitution"][0],
                     m["friction"][0], w.pos, w.vel, w.mass, w.cutoff_radius, w.radius,
                     omega=w.omega, tag=w.tag)
    s.run(120)
    st = s.state()
    f, t = s.forces()
    out = dict(st, force=f, torque=t, rebuilds=np.array(s.thermo()["rebuilds"]))
    for k, v in zip(("owner", "partner", "code"), s.pairs()):
        out[k] = v
    s.close()
    return out


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("bins", [0.0, 1.5, 4.0])
@pytest.mark.parametrize("kind", ["one", "small", "uneven", "poly"])
def test_batch_rows_are_the_same_either_way(kind, bins, prec):
    ws = _systems(kind)
    a, b, c = (_run(ws, prec, mode, bins) for mode in (1, 2, 0))
    assert a["rebuilds"] > 1 and (kind == "one" or len(a["owner"]) > 0)
    for k in a:
        assert np.array_equal(a[k], b[k]) and np.array_equal(a[k], c[k]), k


@pytest.mark.parametrize("phi", [0.1, 0.17, 0.3])
def test_rows_around_two_chunks_of_candidates(phi):
    # cells with about 80, 140 and 240 candidates: up to 128 their rows are written
    # as they are found, beyond from lists
    n = 30000
    w = W.gas_system(n, phi, 0.9, 0.4, seed=8)
    w.pos = W.Stream(12).uniform(3 * n).reshape(-1, 3) * w.hi  # off its lattice
    rows = []
    for mode in (1, 2):
        s = hip.from_workload(w, hip.MIXED, box_exit=False)
        s.set_build_kernel(mode)
        s.bin_neighbor_list()
        rows.append(s.pairs())
        s.close()
    assert len(rows[0][0]) > 0
    for x, y in zip(*rows):
        assert np.array_equal(x, y)
