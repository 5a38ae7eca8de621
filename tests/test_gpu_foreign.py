"""Slot and row fields that someone else rewrites between two calls of a context -- another context's
icf_pack_pcsr, or a copy that the context does not issue -- and that the context then packs itself: it finds them
right already, but its slot maps and the batched layout check were made from others."""
import ctypes

import numpy as np
import pytest

from icflow_amd import _lib, specimens
from icflow_amd.gpu_functionality import CSR, GPUFunctionality
from workloads import H, Pipeline, make_state, small_specimen

pytestmark = pytest.mark.gpu


def _pack(lib, ctx, gf, col, alt, rows, cols):
    _lib.check(lib.icf_pack_pcsr(ctx, alt.p, alt.n, rows.p, cols.p, rows.n - 1, gf.g_ie_pcsr.p, len(col.elastic),
                                 gf.el_elastic_stride, gf.g_icz.p, len(col.czs), gf.cz_stride, None, 0, 0), ctx, "pack")


def _with_block(rows, cols, r, N):
    """The pattern with one more block in row r, at a column that the row lacks."""
    c = next(c for c in range(N - 1, r, -1) if c not in cols[rows[r]:rows[r + 1]])
    at = rows[r] + np.searchsorted(cols[rows[r]:rows[r + 1]], c)
    rows = rows.copy()
    rows[r + 1:] += 1
    return rows, np.insert(cols, at, c).astype(np.int32)


@pytest.mark.parametrize("writer", ["pack", "copy"])
def test_slots_that_others_made_right(specimen_consts, writer):
    col = small_specimen(cells=(5, 4, 4), size=(0.05, 0.04, 0.04), grains=5, seed=9, platens=False)
    p = Pipeline(col, specimen_consts, make_state(col, specimen_consts, seed=10))
    gf, lib, ctx = p.gf, p.gf.lib, p.gf.ctx
    N = gf.csr.N
    other = GPUFunctionality(0)
    # two patterns of the same size whose slots differ from row 1 to row N / 2
    pats = [_with_block(gf.csr.rows, gf.csr.cols, r, N) for r in (1, N // 2)]
    nnz = len(pats[0][1])
    alt = gf.buf("alt", len(col.alt), np.int32)
    alt.upload(np.ascontiguousarray(col.alt, np.int32))
    dev = []
    for k, (rows, cols) in enumerate(pats):
        dev.append((gf.buf("rows%d" % k, N + 1, np.int32), gf.buf("cols%d" % k, nnz, np.int32)))
        dev[k][0].upload(rows)
        dev[k][1].upload(cols)
    vals, rhs = gf.buf("v", 9 * nnz, np.float64), gf.buf("r", 3 * N, np.float64)

    def assembled(k):
        _lib.check(lib.icf_assemble_elems_and_czs(
            ctx, gf.g_ie_pcsr.p, len(col.elastic), gf.el_elastic_stride, gf.g_dcz.p, gf.g_icz.p, len(col.czs),
            gf.cz_stride, gf.g_dn.p, gf.nd_stride, H, vals.p, nnz, rhs.p, N, None, None), ctx, "assemble")
        rows, cols = pats[k]
        r = np.repeat(np.arange(N), np.diff(rows))
        return dict(zip(zip(r.tolist(), cols.tolist()), vals.download(9 * nnz).reshape(-1, 9)))

    def rewritten(k):
        if writer == "pack":
            _pack(lib, other.ctx, gf, col, alt, *dev[k])
            return
        for buf, kept in zip((gf.g_ie_pcsr, gf.g_icz), copies[k]):
            _lib.check(lib.icf_d2d(other.ctx, buf.p, 0, kept.p, 0, 4 * buf.n), other.ctx, "d2d")
        _lib.check(lib.icf_synchronize(other.ctx), other.ctx, "sync")

    copies = []
    for k in range(2):
        _pack(lib, ctx, gf, col, alt, *dev[k])
        copies.append([gf.buf("%s%d" % (n, k), b.n, np.int32) for n, b in (("ie", gf.g_ie_pcsr), ("icz", gf.g_icz))])
        for buf, kept in zip((gf.g_ie_pcsr, gf.g_icz), copies[k]):
            kept.upload(buf.download())
    _pack(lib, ctx, gf, col, alt, *dev[0])
    want = assembled(0)
    for k in (1, 0, 1, 1, 0):
        rewritten(k)
        _pack(lib, ctx, gf, col, alt, *dev[k])
        got = assembled(k)
        for key, x in got.items():
            assert np.array_equal(x, want.get(key, np.zeros(9))), (k, key)
    other.close()
    gf.close()


def test_batched_layout_that_others_broke(specimen_consts):
    col = specimens.lognormal_cubes(3, 3, median_tets=600, min_tets=300, max_tets=1000, sigma=0.5, grains=(3, 5), size=0.01)
    st = specimens.synthetic_state(col, specimen_consts, 8)
    gf = GPUFunctionality(0)
    gf.SetConstants(specimen_consts)
    gf.TransferStaticDataToDevice(col)
    gf.TransferNodesToGPU(st)
    gf.CreateStructure(None)
    gf.TransferPCSR(st)
    lib, ctx, N = gf.lib, gf.ctx, gf.csr.N
    tet, cz, row = specimens.specimen_offsets(col)
    offs = [tet, cz, row, gf.csr.rows[row].astype(np.int32)]
    # the same units with a row of specimen 0 and one of specimen 1 exchanged: as many blocks, but
    # both specimens write into the other's
    base = np.ascontiguousarray(col.alt, np.int32)
    swapped = base.copy()
    swapped[base == row[1] - 1], swapped[base == row[1]] = row[1], row[1] - 1
    other = GPUFunctionality(0)
    sets = []
    for k, a in enumerate((base, swapped)):
        csr = CSR(lib).build(a[col.elastic], a[col.czs])
        assert csr.nnz == gf.csr.nnz
        bufs = [gf.buf("%s%d" % (n, k), len(v), np.int32) for n, v in (("a", a), ("rows", csr.rows), ("cols", csr.cols))]
        for b, v in zip(bufs, (a, csr.rows, csr.cols)):
            b.upload(v)
        sets.append(bufs)
    wl = _lib.IcfWorklist(len(tet) - 1, *[_lib.ptr(v) for v in offs])
    vals, rhs = gf.buf("v", 9 * gf.csr.nnz, np.float64), gf.buf("r", 3 * N, np.float64)
    for k in (0, 1, 0, 1, 1, 0):
        _pack(lib, other.ctx, gf, col, *sets[k])
        _pack(lib, ctx, gf, col, *sets[k])
        r = lib.icf_assemble_batched(ctx, ctypes.byref(wl), gf.g_ie_pcsr.p, gf.el_elastic_stride, gf.g_dcz.p,
                                     gf.g_icz.p, gf.cz_stride, gf.g_dn.p, gf.nd_stride, H, vals.p, rhs.p, None, None)
        assert r == (_lib.ICF_E_INDEX if k else 0), k
    other.close()
    gf.close()
