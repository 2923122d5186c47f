"""Downloads return what was uploaded, value for value, at the sizes where the
copy changes its shape: one wait for everything (LJ up to 32,768 particles, 64
bytes each), then pieces of half a MiB over several host threads."""
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
@pytest.mark.parametrize("n", [1, 65, 32768, 32769, 100003])
def test_downloads_return_the_uploads(n, model, prec):
    st = W.Stream(n)
    dem = model == hip.MODEL_DEM
    pos, vel, omega, f, t = (st.uniform(3 * n).reshape(n, 3) for _ in range(5))
    quat = st.uniform(4 * n).reshape(n, 4)
    mass, rad, cut = (0.5 + st.uniform(n) for _ in range(3))
    tag = np.arange(n, dtype=np.uint32)[::-1].copy()
    kind = (np.arange(n) % 3).astype(np.uint32)
    s = hip.System(model, prec)
    if dem:
        s.set_materials([1e7] * 3, [0.3] * 3, [0.9] * 3, [0.4] * 3)
    s.upload(pos, vel, mass, cut, radius=rad if dem else None, omega=omega if dem else None, tag=tag,
             atype=kind)
    for _ in range(2):  # the second call reuses the staging memory
        got = s.state()
        assert np.array_equal(got["tag"], tag)
        assert np.array_equal(got["pos"], pos) and np.array_equal(got["vel"], vel)
        assert not got["image"].any()
    ty, m, r, c = s.properties()
    assert np.array_equal(ty, kind) and np.array_equal(m, mass) and np.array_equal(c, cut)
    s.set_forces(f, t if dem else None)
    gf, gt = s.forces()
    low = np.float32 if prec == hip.MIXED else np.float64
    assert np.array_equal(gf, f.astype(low).astype(np.float64))
    if dem:
        assert np.array_equal(got["omega"], omega) and np.array_equal(r, rad)
        assert np.array_equal(gt, t.astype(low).astype(np.float64))
        s.upload_quaternions(quat)
        assert np.array_equal(s.state()["quat"], quat)
    s.close()
