"""A download does without the host threads it cannot have: where the system
refuses new threads, the calling thread places every piece."""
import resource
import sys
import threading

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


@pytest.mark.parametrize("n", [32769, 300001])
def test_downloads_without_new_threads(n):
    st = W.Stream(n)
    pos, vel = (st.uniform(3 * n).reshape(n, 3) for _ in range(2))
    s = hip.System(hip.MODEL_LJ)
    s.upload(pos, vel, np.ones(n), np.ones(n))
    s.state()  # everything that is made once is made
    soft, hard = resource.getrlimit(resource.RLIMIT_NPROC)
    resource.setrlimit(resource.RLIMIT_NPROC, (1, hard))
    try:
        try:
            t = threading.Thread(target=lambda: None)
            t.start()
            t.join()
            refused = False
        except RuntimeError:
            refused = True
        got = s.state() if refused else None
    finally:
        resource.setrlimit(resource.RLIMIT_NPROC, (soft, hard))
    s.close()
    if not refused:
        pytest.skip("this user's threads are not limited")
    assert np.array_equal(got["pos"], pos) and np.array_equal(got["vel"], vel)
    assert np.array_equal(got["tag"], np.arange(n)) and not got["image"].any()
