"""The row build of dense grids, over what it chooses between: wavefronts per
cell, candidates in registers or from memory, row layouts, members of one kind
or two. The one-lane-per-member kernel takes any grid and is the reference:
same rows, so the same pairs in the same order and bitwise the same forces."""
import sys

import numpy as np
import pytest

from mddem_amd import hip
from mddem_amd import workloads as W
from tests.helpers import canonical_pairs, oracle_from_workload
from tests.test_gpu_parity import _dense_dem, _oracle_rebuild, _perturbed_lj

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    print(f"\n[gpu case] {request.node.name}", flush=True)
    sys.stdout.flush()
    yield


def _face_atoms(rho):
    """Atoms a rounding error from a face of the box: at these densities some
    land in a bin of the image layer, or images in a bin of the box, so that
    bins hold particles and images."""
    w = W.lj_fcc(ncell=7, rho=rho)
    w.pos = w.pos + (W.Stream(11).uniform(3 * w.n).reshape(-1, 3) - 0.5) * 0.05
    L = w.hi - w.lo
    w.pos = np.mod(w.pos, L)
    for d in range(3):
        w.pos[w.pos[:, d] > L[d] - 0.03, d] = np.nextafter(L[d], 0.0)
        w.pos[w.pos[:, d] < 0.03, d] = 1e-18
    reach = 2.0 * 1.25 * w.skin_fraction
    bins = np.floor(L / reach)
    bs = L / bins
    layers = np.ceil((reach + 0.3) / bs) + np.ceil(reach / bs)
    cell = lambda x: np.floor((x + bs * layers) * (1.0 / bs)) - layers
    high, low = cell(np.nextafter(L, 0.0)), cell(np.full(3, 1e-18) + L)
    assert np.any(high == bins) or np.any(low < bins)
    return w


def _case(name):
    if name.startswith("lj_"):  # 216 cells in the box, 850 .. 10,240, more
        return _perturbed_lj(n=int(name[3:]))
    w = _perturbed_lj(n=11)
    if name == "wide_bins":  # above 640 candidates per cell
        w.bin_size = 3.6
    elif name == "huge_bins":  # above 1,024
        w.bin_size = 5.0
    elif name == "long_rows":  # few lists fit at once
        w.cutoff_radius = np.full(w.n, 2.2)
    elif name.startswith("faces"):
        return _face_atoms(0.01 * int(name[6:]))
    elif name == "poly":
        w = _dense_dem(n=1500, seed=7)
        st = W.Stream(9)
        w.radius = w.radius * (0.8 + 0.2 * st.uniform(w.n))
        w.cutoff_radius = w.radius.copy()
    return w


def _rows(w, mode, lanes=None):
    s = hip.from_workload(w, hip.FP64)
    if lanes is not None:
        s.set_force_lanes(lanes)
    s.set_build_kernel(mode)
    s.bin_neighbor_list()
    pairs = s.pairs()
    if w.model == "lj":
        s.lj_force()
    else:
        s.hertz_mindlin_contact_force()
    out = (*pairs, s.state()["tag"], *s.forces())
    s.close()
    return out


CASES = ["lj_6", "lj_10", "lj_18", "lj_40", "wide_bins", "huge_bins", "long_rows", "faces_90", "faces_84",
         "poly"]


@pytest.mark.parametrize("name", CASES)
def test_rows_are_those_of_member_lanes(name):
    w = _case(name)
    a, b = _rows(w, 1), _rows(w, 2)
    assert len(a[0]) > 0
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("lanes", [0, 1, 2, 3])
@pytest.mark.parametrize("name", ["lj_6", "wide_bins", "faces_90", "faces_84", "poly"])
def test_every_row_layout_is_filled_alike(name, lanes):
    w = _case(name)
    for x, y in zip(_rows(w, 1, lanes), _rows(w, 2, lanes)):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("name", ["lj_10", "wide_bins", "faces_90", "faces_84", "poly"])
def test_pairs_are_the_oracles(name):
    w = _case(name)
    o = oracle_from_workload(w)
    _oracle_rebuild(o)
    assert np.array_equal(canonical_pairs(*_rows(w, 1)[:3]), canonical_pairs(*o.pairs()))
