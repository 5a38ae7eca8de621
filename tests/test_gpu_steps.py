"""Broad phase (icf_broad_phase) against all pairs: tets that touch exactly, ranges of sizes from a
fraction of a grid cell to the whole scene, scenes far from the origin and so far that positions
keep few digits, points, one cell and thousands, with one context going from small scenes to large ones."""
import ctypes

import numpy as np
import pytest

from icflow_amd import _lib
from icflow_amd.gpu_functionality import GPUFunctionality

pytestmark = pytest.mark.gpu


def overlapping(x, ids, exclude):
    """Pairs a < b of tets x[t, 4, 3] whose 12 k-DOP extents overlap and, if asked, share no node."""
    p = [x[..., k] for k in range(3)]
    p = p + [p[0] + p[1], p[0] + p[2], p[1] + p[2], p[0] - p[1], p[0] - p[2], p[1] - p[2],
             p[0] + p[1] - p[2], p[0] + p[2] - p[1], p[1] + p[2] - p[0]]
    lo, hi = np.array([q.min(1) for q in p]), np.array([q.max(1) for q in p])
    out = []
    for a in range(len(x) - 1):
        hit = ((lo[:, a, None] <= hi[:, a + 1:]) & (hi[:, a, None] >= lo[:, a + 1:])).all(0)
        if exclude:
            hit &= ~(ids[a][:, None, None] == ids[a + 1:][None]).any((0, 2))
        b = np.nonzero(hit)[0] + a + 1
        out.append(np.stack([np.full(len(b), a), b], 1))
    return np.concatenate(out) if out else np.zeros((0, 2), int)


def test_pairs_match_all_pairs():
    rng = np.random.default_rng(11)
    gf = GPUFunctionality(0)
    lib, ctx = gf.lib, gf.ctx
    for n, span, size, lattice, offset in (
            (1, 1, 1, 0, 0), (2, 0, 0, 0, 0), (65, 1, 1, 8, 0), (300, 6, 1, 4, 0), (1200, 9, 1, 16, 0),
            (1200, 40, 1, 0, 0), (700, 8, 1, 2, -3e5), (700, 8, 1, 0, 1e9), (500, 6, 1, 0, 3e12),
            (400, 5, 1e-3, 0, 4e12), (900, 300, 1, 0, 0), (1200, 3, 3, 0, 0), (40, 2, 0, 2, 0)):
        nodes = max(4, 3 * n)                                # nodes are shared now and then
        corner = span * rng.random((n, 1, 3))
        t = corner + size * rng.random((n, 4, 3)) * rng.choice([1, 1, 1, 0.05], (n, 1, 1))
        if lattice:
            t = np.round(t * lattice) / lattice              # many planes coincide
        x = np.zeros((nodes, 3))
        ids = np.arange(4 * n).reshape(n, 4) % nodes
        x[ids.ravel()] = t.reshape(-1, 3)
        x += offset
        ids = ids.astype(np.int32)
        ns, es = nodes + 3, n + 2
        dn, ie = np.zeros((18, ns)), np.zeros((5, es), np.int32)
        dn[15:18, :nodes] = x.T
        ie[:4, :n] = ids.T
        d_dn, d_ie = gf.buf("dn", dn.size, np.float64), gf.buf("ie", ie.size, np.int32)
        d_dn.upload(dn.ravel())
        d_ie.upload(ie.ravel())
        for exclude in (1, 0):
            ref = overlapping(x[ids], ids, exclude)
            d_pairs = gf.buf("pairs", 2 * len(ref) + 2, np.int32)
            num = ctypes.c_longlong()
            for _ in range(2):
                _lib.check(lib.icf_broad_phase(ctx, d_dn.p, ns, d_ie.p, es, n, exclude, d_pairs.p, len(ref) + 1,
                                               ctypes.byref(num)), ctx, "broad_phase")
                assert num.value == len(ref), (n, span, offset, exclude)
                assert np.array_equal(d_pairs.download(2 * len(ref)).reshape(-1, 2), ref), (n, span, offset)
    # a node id out of range, then positions that are not finite, are refused; the next call works
    d_ie.upload(np.where(np.arange(ie.size) == 1, ns, ie.ravel()).astype(np.int32))
    args = (ctx, d_dn.p, ns, d_ie.p, es, n, 0, d_pairs.p, len(ref) + 1, ctypes.byref(num))
    assert lib.icf_broad_phase(*args) == _lib.ICF_E_INDEX
    d_ie.upload(ie.ravel())
    d_dn.upload(np.where(dn == dn[15, 2], -np.inf, dn).ravel())
    assert lib.icf_broad_phase(*args) == _lib.ICF_E_INVALID
    d_dn.upload(dn.ravel())
    assert lib.icf_broad_phase(*args) == 0 and num.value == len(ref)
    gf.close()
