"""Broad phase (icf_broad_phase) on scenes whose candidate pairs crowd into a few grid cells: one large
tet sets the cells' size, thousands of tiny ones lie so close together that the search's steps do
not tell them apart, and hardly any of them overlap."""
import ctypes

import numpy as np
import pytest

from icflow_amd import _lib, specimens
from icflow_amd.gpu_functionality import GPUFunctionality

pytestmark = pytest.mark.gpu

CLUSTERS = 8
FRACTION = (0.06, 0.22, 0.54)             # of a step, so that no plane of a cluster crosses one


def _scene(n):
    """Tiny tets on a lattice in each of the cells 0 to 7 along x, the last three of a cluster where its
    first three are; a tiny tet at the origin; a tet of size 1 beyond them.  Returns positions and the pairs."""
    cs = 1.000001                           # the cell for extents of 1
    step, e = cs / 2048, 28
    i = np.arange(n - 3)
    at = np.stack([i % e, i // e % e, i // (e * e)], 1) * 1.6e-6
    at = np.concatenate([at, at[:3]])
    # within one step in each of the 12 directions
    base = step * np.array(FRACTION)
    x = np.concatenate([at + base + [k * cs, 0, 0] for k in range(CLUSTERS)] + [np.zeros((1, 3))])
    tiny = 1e-7 * np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
    x = x[:, None] + tiny
    big = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]]) + [9.5, 0, 0]
    x = np.concatenate([x, big[None]])
    pairs = [(k * n + j, k * n + n - 3 + j) for k in range(CLUSTERS) for j in range(3)]
    return x, np.array(pairs)


def _search(gf, x, ids, room):
    n, ns, es = len(ids), len(x), len(ids)
    dn, ie = np.zeros((18, ns)), np.zeros((5, es), np.int32)
    dn[15:18] = x.T
    ie[:4] = ids.T
    d_dn, d_ie = gf.buf("dn%d" % n, dn.size, np.float64), gf.buf("ie%d" % n, ie.size, np.int32)
    d_dn.upload(dn.ravel())
    d_ie.upload(ie.ravel())
    d_pairs, num = gf.buf("pairs", 2 * room, np.int32), ctypes.c_longlong()
    for _ in range(2):
        _lib.check(gf.lib.icf_broad_phase(gf.ctx, d_dn.p, ns, d_ie.p, es, n, 1, d_pairs.p, room, ctypes.byref(num)),
                   gf.ctx, "broad_phase")
        yield d_pairs.download(2 * room).reshape(-1, 2)[:num.value]


# 2.2e8 pairs that the steps do not tell apart, which the buffer holds if they are spread over its regions,
# and 1.8e9, which it does not
@pytest.mark.parametrize("n", [7400, 21000])
def test_crowded_cells(n):
    gf = GPUFunctionality(0)
    for count in (10, n):                   # the small scene sizes the second one's launches
        x, want = _scene(count)
        for got in _search(gf, x.reshape(-1, 3), np.arange(4 * len(x)).reshape(-1, 4), 4096):
            assert np.array_equal(got, want), count
    gf.close()


def test_first_search_of_a_context(specimen_consts):
    """More candidates than a new context's buffer takes: the tets of a cell may lie in another order in
    the second search, whose regions have to hold what the first one counted."""
    col = specimens.make_specimen((3, 3, 3), (0.0075,) * 3, 2, 1, platens=(2, 2)).finalize()
    for seed in range(150):
        st = specimens.synthetic_state(col, specimen_consts, seed, platen_dz=0.3 * 0.0025)
        gf, want = GPUFunctionality(0), None
        for got in _search(gf, col.x0 + st.un, col.surf, 10000):
            want = got if want is None else want
            assert len(want) > 0 and np.array_equal(got, want)
        gf.close()
