"""Broad phase (icf_broad_phase) on scenes whose candidate pairs crowd into a few grid cells: one large
tet sets the cells' size, thousands of tiny ones lie so close together that the search's steps do
not tell them apart, and hardly any of them overlap."""
import ctypes

import numpy as np
import pytest

from icflow_amd import _lib
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


def _search(gf, x, room):
    n = len(x)
    ns, es = 4 * n, n
    dn, ie = np.zeros((18, ns)), np.zeros((5, es), np.int32)
    dn[15:18] = x.reshape(-1, 3).T
    ie[:4] = np.arange(4 * n).reshape(n, 4).T
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
        for got in _search(gf, x, 4096):
            assert np.array_equal(got, want), count
    gf.close()
