"""A context's first download is read another way than the later ones: forces
and properties come back as uploaded whichever call is the first."""
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


@pytest.mark.parametrize("prec", [hip.MIXED, hip.FP64])
@pytest.mark.parametrize("model", [hip.MODEL_LJ, hip.MODEL_DEM])
@pytest.mark.parametrize("n", [1, 63, 65, 40001])
def test_any_call_can_be_the_first(n, model, prec):
    st = W.Stream(n)
    dem = model == hip.MODEL_DEM
    pos, vel, f, t = (st.uniform(3 * n).reshape(n, 3) for _ in range(4))
    mass, rad, cut = (0.5 + st.uniform(n) for _ in range(3))
    kind = (np.arange(n) % 3).astype(np.uint32)
    low = np.float32 if prec == hip.MIXED else np.float64
    for first in ("forces", "properties", "state"):
        s = hip.System(model, prec)
        if dem:
            s.set_materials([1e7] * 3, [0.3] * 3, [0.9] * 3, [0.4] * 3)
        s.upload(pos, vel, mass, cut, radius=rad if dem else None, atype=kind)
        s.set_forces(f, t if dem else None)
        for call in (first, first, "forces", "properties", "state"):
            if call == "forces":
                gf, gt = s.forces()
                assert np.array_equal(gf, f.astype(low).astype(np.float64))
                assert not dem or np.array_equal(gt, t.astype(low).astype(np.float64))
            elif call == "properties":
                ty, m, r, c = s.properties()
                assert np.array_equal(ty, kind) and np.array_equal(m, mass)
                assert np.array_equal(c, cut) and (not dem or np.array_equal(r, rad))
            else:
                got = s.state()
                assert np.array_equal(got["pos"], pos) and np.array_equal(got["vel"], vel)
        s.close()
