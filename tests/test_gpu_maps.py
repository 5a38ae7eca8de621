"""Slot maps built anew in their own buffers: unit counts and slots that change from call to call
over the same arrays -- fewer and more units, keys beyond what earlier maps counted, runs of keys
across the tiles of the scan -- each against the oracle."""
import ctypes

import numpy as np
import pytest

from conftest import rel_err
from icflow_amd import _lib
from workloads import H, Pipeline, make_state, small_specimen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,grains", [((2, 1, 1), 2), ((6, 5, 4), 6)])
def test_maps_follow_changing_units(orc, specimen_consts, cells, grains):
    col = small_specimen(cells=cells, size=tuple(0.01 * c for c in cells), grains=grains, seed=3, platens=False)
    p = Pipeline(col, specimen_consts, make_state(col, specimen_consts, seed=4))
    gf, lib, ctx = p.gf, p.gf.lib, p.gf.ctx
    T, C, N, nnz = len(col.elastic), len(col.czs), gf.csr.N, gf.csr.nnz
    es, cs, ns = gf.el_elastic_stride, gf.cz_stride, gf.nd_stride
    orc.set_constants(specimen_consts)
    top = 9000
    g_A, g_b = gf.buf("A", 9 * (nnz + top), np.float64), gf.buf("b", 3 * N, np.float64)
    # units taken (share of all), slots moved up by so much; the last keys fill a scan tile exactly,
    # then one more and one less
    tile = 2048 - nnz % 2048
    for share, shift in ((1.0, 0), (0.01, 0), (0.5, tile), (1.0, tile + 1), (0.3, tile - 1), (1.0, top), (1.0, 0)):
        nE, nC, n = max(1, int(share * T)), max(1, int(share * C)), nnz + shift
        ie, icz, dcz, dn = gf.c_ie_pcsr.copy(), gf.c_icz.copy(), gf.c_dcz.copy(), gf.c_dn.copy()
        for a, lo, hi in ((ie, 4 * es, 20 * es), (icz, 10 * cs, 46 * cs)):
            a[lo:hi] = np.where(a[lo:hi] >= 0, a[lo:hi] + shift, a[lo:hi])
        for buf, a in ((gf.g_ie_pcsr, ie), (gf.g_icz, icz), (gf.g_dcz, dcz), (gf.g_dn, dn)):
            buf.upload(a)
        ref = dn.copy()
        A, b = np.zeros(9 * n), np.zeros(3 * N)
        orc.elem_force(ie.copy(), ref, H, A, b, nE, es, ns)
        orc.cz_force(dcz.copy(), icz.copy(), ref, A, b, H, nC, cs, ns)
        args = (gf.g_ie_pcsr.p, nE, es, gf.g_dcz.p, gf.g_icz.p, nC, cs, gf.g_dn.p, ns, H, g_A.p)
        if nE == T:                          # every row has its tets: exact sizes are known
            _lib.check(lib.icf_assemble_elems_and_czs(ctx, *args, n, g_b.p, N, None, None), ctx, "assemble")
            one = g_A.download(9 * n), g_b.download(3 * N)
            assert rel_err(one[0], A) <= 1e-9 and rel_err(one[1], b) <= 1e-9
            assert rel_err(gf.g_dn.download()[12 * ns:15 * ns], ref[12 * ns:15 * ns]) <= 1e-9
        # ... and added up by the single calls, whose maps count keys as they need
        for buf, a in ((gf.g_icz, icz), (gf.g_dcz, dcz), (gf.g_dn, dn)):
            buf.upload(a)
        g_A.zero()
        g_b.zero()
        _lib.check(lib.icf_elem_force(ctx, gf.g_ie_pcsr.p, gf.g_dn.p, H, g_A.p, g_b.p, nE, es, ns), ctx, "elem")
        _lib.check(lib.icf_cz_force(ctx, gf.g_dcz.p, gf.g_icz.p, gf.g_dn.p, g_A.p, g_b.p, H, nC, cs, ns), ctx, "cz")
        assert rel_err(g_A.download(9 * n), A) <= 1e-9 and rel_err(g_b.download(3 * N), b) <= 1e-9
    # a slot beyond the declared size is refused, and the next call with the right size works
    dmg = ctypes.c_int()
    r = lib.icf_assemble_elems_and_czs(ctx, gf.g_ie_pcsr.p, T, es, gf.g_dcz.p, gf.g_icz.p, C, cs, gf.g_dn.p, ns, H,
                                       g_A.p, nnz - 1, g_b.p, N, ctypes.byref(dmg), None)
    assert r == _lib.ICF_E_INDEX
    gf.g_dn.upload(dn)
    gf.g_dcz.upload(dcz)
    _lib.check(lib.icf_assemble_elems_and_czs(ctx, gf.g_ie_pcsr.p, T, es, gf.g_dcz.p, gf.g_icz.p, C, cs, gf.g_dn.p, ns,
                                              H, g_A.p, nnz, g_b.p, N, None, None), ctx, "assemble")
    assert rel_err(g_A.download(9 * nnz), A) <= 1e-9
    gf.close()
