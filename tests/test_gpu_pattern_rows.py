"""Rows that impacts add to a kept pattern (icf_build_pattern), against all pairs' keys: rows with
few and many new columns (one node in every impact), repeated pairs, more candidates than the
workgroup's buffer, row counts around a workgroup's, no static part."""
import ctypes

import numpy as np
import pytest

from icflow_amd import _lib
from icflow_amd.gpu_functionality import GPUFunctionality

pytestmark = pytest.mark.gpu


def pattern(alt, units, N):
    """Rows and columns of c >= r over each element's and CZ's pairs and c > r over each impact's."""
    keys = [np.zeros(0, np.int64)]
    for u, strict in zip(units, (0, 0, 1)):
        i, j = np.divmod(np.arange(u.shape[1] ** 2), u.shape[1])
        r, c = alt[u][:, i].astype(np.int64), alt[u][:, j].astype(np.int64)
        keys.append((r * N + c)[(r >= 0) & (c >= r + strict)])
    keys = np.unique(np.concatenate(keys))
    return np.searchsorted(keys, np.arange(N + 1) * N), keys % N


@pytest.mark.parametrize("nodes,tets,czs,impacts,hub", [
    (9, 1, 0, 1, 0.0), (256, 300, 20, 64, 0.0), (257, 300, 0, 4000, 0.0), (255, 0, 0, 500, 0.5),
    (3000, 9000, 700, 20, 1.0), (3000, 9000, 700, 2500, 0.6), (66000, 2000, 100, 900, 0.2)])
def test_impact_rows_match_all_pairs(nodes, tets, czs, impacts, hub):
    rng = np.random.default_rng(nodes + impacts)
    alt = np.arange(nodes, dtype=np.int32)
    alt[(rng.random(nodes) < 0.1) & (alt != 3)] = -1
    alt[alt >= 0] = np.arange((alt >= 0).sum())
    N = int((alt >= 0).sum())
    units = [rng.integers(0, nodes, (n, k)).astype(np.int32) for n, k in ((tets, 4), (czs, 6), (impacts, 4))]
    units[2][rng.random(impacts) < hub, 0] = 3
    gf = GPUFunctionality(0)
    lib, ctx = gf.lib, gf.ctx
    offs, bufs, strides = (0, 4, 0), [], []
    for k, u in enumerate(units):
        stride = max(len(u), 1) + 3
        a = np.full((52, stride), -1, np.int32)
        a[offs[k]:offs[k] + u.shape[1], :len(u)] = u.T
        b = gf.buf(f"u{k}", a.size, np.int32)
        b.upload(a.ravel())
        bufs.append(b)
        strides.append(stride)
    d_alt = gf.buf("alt", nodes, np.int32)
    d_alt.upload(alt)
    cap = 10 * tets + 21 * czs + 6 * impacts + 1
    d_rows, d_cols = gf.buf("rows", N + 1, np.int32), gf.buf("cols", cap, np.int32)

    def build(nimp, room):
        nnz = ctypes.c_int()
        r = lib.icf_build_pattern(ctx, d_alt.p, nodes, bufs[0].p, tets, strides[0], bufs[1].p, czs, strides[1],
                                  bufs[2].p, nimp, strides[2], N, d_rows.p, d_cols.p, room, ctypes.byref(nnz))
        return r, nnz.value

    for nimp in (impacts, 0, impacts // 2, impacts):        # the static part is kept after the first
        rows, cols = pattern(alt, (units[0], units[1], units[2][:nimp]), N)
        r, nnz = build(nimp, cap)
        assert r == 0 and nnz == rows[-1]
        assert np.array_equal(d_rows.download(N + 1), rows) and np.array_equal(d_cols.download(nnz), cols)
        if nnz:                                             # refused, and nothing is written
            d_rows.upload(np.full(N + 1, -5, np.int32))
            r, n = build(nimp, nnz - 1)
            assert r == _lib.ICF_E_CAPACITY and n == nnz and (d_rows.download(N + 1) == -5).all()
    bad = units[2].copy()
    bad[-1, 2] = nodes
    a = np.full((52, strides[2]), -1, np.int32)
    a[:4, :impacts] = bad.T
    bufs[2].upload(a.ravel())
    assert build(impacts, cap)[0] == _lib.ICF_E_INDEX
    assert build(impacts - 1, cap)[0] == 0                  # the last impact alone is out of range
    gf.close()
