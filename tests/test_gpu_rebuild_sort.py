"""The rebuild's sort and images at the edges of their tiles: particle counts
around the wavefront, the workgroup and the 1,024 particles that share an image
total; cell counts around one scan tile (4,096) and around the largest grid
scanned in one launch (131,072); many particles in one cell. Particle order,
pairs and image shifts must be the oracle's."""
import sys

import numpy as np
import pytest

from mddem_amd import hip
from mddem_amd import workloads as W
from tests.helpers import canonical_pairs, oracle_from_workload
from tests.test_gpu_parity import _oracle_rebuild

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


def _random(n, bins, seed, pile=0):
    """n atoms at random in a box of that many bins a side (the grid has six
    more along each axis); the first `pile` of them inside one bin."""
    w = W.lj_fcc(ncell=3)
    st = W.Stream(seed)
    L = np.array(bins) * 1.0005 * 2.0 * 1.25 * w.skin_fraction
    pos = st.uniform(3 * n).reshape(n, 3) * L
    pos[:pile] = 1e-3 * L + 0.9 * st.uniform(3 * pile).reshape(pile, 3) * (L / np.array(bins))
    w.lo, w.hi, w.pos = np.zeros(3), L, pos
    w.vel = np.zeros((n, 3))
    w.mass = np.ones(n)
    w.cutoff_radius = np.full(n, 1.25)
    return w


CASES = {
    "n1": (1, (3, 3, 3), 0),
    "n63": (63, (3, 3, 3), 0),
    "n257": (257, (3, 4, 3), 0),
    "n1023": (1023, (4, 4, 4), 0),
    "n1024": (1024, (4, 4, 4), 0),
    "n1025": (1025, (4, 4, 4), 0),
    "n4097": (4097, (6, 5, 6), 0),
    "cells4096": (3000, (10, 10, 10), 0),
    "cells4352": (3000, (11, 10, 10), 0),
    "cells131072": (9000, (58, 58, 26), 0),
    "cells135168": (9000, (58, 58, 27), 0),
    "pile": (2000, (5, 5, 5), 300),
}


@pytest.mark.parametrize("name", list(CASES))
def test_sort_and_images_are_the_oracles(name):
    n, bins, pile = CASES[name]
    w = _random(n, bins, seed=100 + n, pile=pile)
    o = oracle_from_workload(w)
    _oracle_rebuild(o)
    s = hip.from_workload(w, hip.FP64)
    # twice: the second sort starts from sorted particles and used counters
    for _ in range(2):
        s.bin_neighbor_list()
        assert np.array_equal(s.state()["tag"], o.atoms()["tag"][:n])
        got, ref = canonical_pairs(*s.pairs()), canonical_pairs(*o.pairs())
        assert np.array_equal(got, ref)
    s.close()
