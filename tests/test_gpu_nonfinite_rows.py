"""A particle whose position is not finite has no neighbors and leaves the
others' rows as they are without it (bin_neighbor_list, neighbor.rs:810-1080:
no distance to it is below the cutoff, its own included)."""
import sys

import numpy as np
import pytest

from mddem_amd import hip
from mddem_amd import workloads as W
from tests.helpers import canonical_pairs

pytestmark = pytest.mark.gpu

BAD = {"nan": (np.nan, np.nan, np.nan), "nan_y": (1.0, np.nan, 1.0), "inf": (np.inf, 1.0, 1.0),
       "-inf": (1.0, 1.0, -np.inf)}


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


def _pairs(s):
    s.set_build_kernel(1)  # a wavefront per cell
    s.bin_neighbor_list()
    a, b, code = s.pairs()
    return a, b, canonical_pairs(a, b, code)


@pytest.mark.parametrize("where", list(BAD))
@pytest.mark.parametrize("name", ["lj_6", "lj_10", "lj_18", "poly"])
def test_rows_of_the_others_stay(name, where):
    w = W.lj_fcc(ncell=6 if name == "poly" else int(name[3:]), thermostat=False)
    if name == "poly":
        w.cutoff_radius = w.cutoff_radius * (0.9 + 0.1 * W.Stream(4).uniform(w.n))
    k = w.n // 2
    keep = np.arange(w.n) != k

    def system(pos, sel):
        s = hip.System(hip.MODEL_LJ)
        s.set_box(w.lo, w.hi, w.periodic)
        s.set_neighbor(w.skin_fraction, w.bin_size, 0, True, 1000, True)
        s.upload(pos[sel], w.vel[sel], w.mass[sel], w.cutoff_radius[sel], tag=w.tag[sel])
        return s

    ref = system(w.pos, keep)
    pos = w.pos.copy()
    pos[k] = BAD[where]
    s = system(pos, np.ones(w.n, bool))
    want, (a, b, got) = _pairs(ref)[2], _pairs(s)
    assert len(want) > 0 and not np.any((a == k) | (b == k))
    assert np.array_equal(got, want)
    ref.close()
    s.close()


@pytest.mark.parametrize("build", [1, 2])
@pytest.mark.parametrize("where", list(BAD))
def test_a_bad_system_of_a_batch_leaves_the_rest(where, build):
    ws = [W.gas_system(200 + 50 * k, 0.25, 0.9, 0.4, seed=70 + k) for k in range(3)]

    def run(bad):
        s = hip.System(hip.MODEL_DEM, hip.FP64)
        s.set_neighbor(1.1, 0.0, 0, True, 1000, True)
        s.set_dt(ws[0].dt)
        s.set_build_kernel(build)
        s.set_rebuild_on_box_exit(False)  # an infinite position is outside at every step
        for k, w in enumerate(ws):
            pos = w.pos.copy()
            if bad and k == 1:
                pos[7] = BAD[where]
            m = w.materials
            s.add_system(w.lo, w.hi, m["youngs"][0], m["poisson"][0], m["restitution"][0],
                         m["friction"][0], pos, w.vel * 20.0, w.mass, w.cutoff_radius, w.radius,
                         omega=w.omega, tag=w.tag)
        s.run(40)
        st = s.state()
        out = [{q: v[f:f + n] for q, v in st.items()} for f, n in map(s.system_range, (0, 2))]
        s.close()
        return out

    for good, got in zip(run(False), run(True)):
        for q in good:
            assert np.array_equal(good[q], got[q]), q
