"""Distinct (node, tet) tuples of the candidate pairs' masks in first-occurrence order (icf_nl2set),
against the masks taken one by one: numbers of pairs around a workgroup's and beyond a group of
256 of them, empty and full masks, repeated tuples within a pair and far apart, more tuples than the
first table holds, and calls after larger and smaller ones."""
import ctypes

import numpy as np
import pytest

from icflow_amd import _lib
from icflow_amd.gpu_functionality import GPUFunctionality

pytestmark = pytest.mark.gpu


def tuples(masks, pairs, ie):
    i, s = np.nonzero((masks[:, None] >> np.arange(8)) & 1)
    a, b = pairs[i].T
    node = np.where(s < 4, ie[s % 4, b], ie[s % 4, a]).astype(np.int64)
    key = node << 32 | np.where(s < 4, a, b)
    return key[np.sort(np.unique(key, return_index=True)[1])]


def test_tuples_match_masks():
    rng = np.random.default_rng(5)
    gf = GPUFunctionality(0)
    lib, ctx = gf.lib, gf.ctx
    for n, tets, density in ((1, 2, 1.0), (255, 30, 0.5), (256, 1, 1.0), (257, 4000, 1.0), (3000, 100000, 1.0),
                             (70000, 900, 0.02), (70000, 30000, 0.3), (5, 40, 0.0), (1000, 50000, 0.9)):
        stride = tets + 5
        ie = np.full((4, stride), -1, np.int32)
        ie[:, :tets] = rng.integers(0, max(2, tets // 4), (4, tets))
        pairs = rng.integers(0, tets, (n, 2)).astype(np.int32)
        masks = np.where(rng.random(n) < density, rng.integers(1, 256, n), 0).astype(np.int32)
        narrow = np.stack([masks | 0x100, pairs[:, 1]], 1).astype(np.int32)   # only the low byte counts
        ref = tuples(masks, pairs, ie)
        ts = len(ref) + 3
        d_ie, d_pairs, d_masks = (gf.buf(k, a.size, np.int32) for k, a in (("ie", ie), ("p", pairs), ("m", narrow)))
        for d, a in ((d_ie, ie), (d_pairs, pairs), (d_masks, narrow)):
            d.upload(np.ascontiguousarray(a).ravel())
        d_nl2 = gf.buf("nl2", 4 * ts, np.int32)

        def call(room):
            d_nl2.upload(np.full(4 * ts, -9, np.int32))
            num = ctypes.c_int()
            r = lib.icf_nl2set(ctx, d_masks.p, d_pairs.p, n, d_ie.p, stride, d_nl2.p, room, ctypes.byref(num))
            return r, num.value, d_nl2.download(4 * ts)

        r, num, got = call(ts)
        assert r == 0 and num == len(ref), (n, tets)
        assert np.array_equal(got[:num], ref >> 32) and np.array_equal(got[ts:ts + num], ref & 0xffffffff)
        assert (got[num:ts] == -9).all() and (got[ts + num:] == -9).all()
        if num > 1:
            r, k, got = call(num - 1)
            assert r == _lib.ICF_E_CAPACITY and k == num
            assert np.array_equal(got[:num - 1], ref[:-1] >> 32)
    gf.close()
