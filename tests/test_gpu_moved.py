"""Slots that change between calls over the same units: moved apart and back in order (the map's
offsets alone change), permuted, two made one, dropped, and one beyond the blocks declared, each against
the oracle."""
import ctypes

import numpy as np
import pytest

from conftest import rel_err
from icflow_amd import _lib
from workloads import H, Pipeline, make_state, small_specimen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,grains", [((2, 1, 1), 2), ((7, 5, 4), 6)])
def test_assembly_follows_moved_slots(orc, specimen_consts, cells, grains):
    col = small_specimen(cells=cells, size=tuple(0.01 * c for c in cells), grains=grains, seed=5, platens=False)
    p = Pipeline(col, specimen_consts, make_state(col, specimen_consts, seed=6))
    gf, lib, ctx = p.gf, p.gf.lib, p.gf.ctx
    T, C, N, nnz = len(col.elastic), len(col.czs), gf.csr.N, gf.csr.nnz
    es, cs, ns = gf.el_elastic_stride, gf.cz_stride, gf.nd_stride
    orc.set_constants(specimen_consts)
    rng = np.random.default_rng(7)
    apart = np.cumsum(rng.integers(1, 4, nnz)) - 1                # in order, empty blocks between
    tight = np.arange(nnz)
    jump = tight + 3000 * (tight >= nnz // 2)                     # over a tile of the scan
    perm = rng.permutation(nnz)
    swap = apart.copy()
    swap[[0, nnz - 1]] = swap[[nnz - 1, 0]]
    one = tight.copy()
    one[nnz // 2] = one[nnz // 2 - 1]                             # two blocks' contributions in one
    less = np.where(tight == nnz // 3, -1, tight)                 # a block's contributions dropped
    top = max(int(m.max()) for m in (apart, jump)) + 1
    g_A, g_b = gf.buf("A", 9 * top, np.float64), gf.buf("b", 3 * N, np.float64)
    for name, m in (("tight", tight), ("apart", apart), ("tight", tight), ("jump", jump), ("perm", perm),
                    ("apart", apart), ("swap", swap), ("tight", tight), ("one", one), ("tight", tight), ("less", less),
                    ("jump", jump)):
        n = int(m.max()) + 1
        ie, icz, dcz, dn = gf.c_ie_pcsr.copy(), gf.c_icz.copy(), gf.c_dcz.copy(), gf.c_dn.copy()
        for a, lo, hi in ((ie, 4 * es, 20 * es), (icz, 10 * cs, 46 * cs)):
            a[lo:hi] = np.where(a[lo:hi] >= 0, m[np.clip(a[lo:hi], 0, nnz - 1)], a[lo:hi])
        for buf, a in ((gf.g_ie_pcsr, ie), (gf.g_icz, icz), (gf.g_dcz, dcz), (gf.g_dn, dn)):
            buf.upload(a)
        ref = dn.copy()
        A, b = np.zeros(9 * n), np.zeros(3 * N)
        orc.elem_force(ie.copy(), ref, H, A, b, T, es, ns)
        orc.cz_force(dcz.copy(), icz.copy(), ref, A, b, H, C, cs, ns)
        args = (gf.g_ie_pcsr.p, T, es, gf.g_dcz.p, gf.g_icz.p, C, cs, gf.g_dn.p, ns, H, g_A.p)
        g_A.upload(np.full(9 * top, np.nan))
        _lib.check(lib.icf_assemble_elems_and_czs(ctx, *args, n, g_b.p, N, None, None), ctx, name)
        assert rel_err(g_A.download(9 * n), A) <= 1e-9 and rel_err(g_b.download(3 * N), b) <= 1e-9, name
    # a block too few: refused, nothing is written, and the next call is whole again
    for buf, a in ((gf.g_ie_pcsr, gf.c_ie_pcsr), (gf.g_icz, gf.c_icz), (gf.g_dcz, dcz), (gf.g_dn, dn)):
        buf.upload(a)
    g_A.upload(np.full(9 * top, -7.0))
    assert lib.icf_assemble_elems_and_czs(ctx, *args, nnz - 1, g_b.p, N, None, None) == _lib.ICF_E_INDEX
    assert (g_A.download(9 * top) == -7.0).all()
    _lib.check(lib.icf_assemble_elems_and_czs(ctx, *args, nnz, g_b.p, N, None, None), ctx, "whole")
    A = np.zeros(9 * nnz)
    orc.elem_force(gf.c_ie_pcsr.copy(), dn.copy(), H, A, b, T, es, ns)
    orc.cz_force(dcz.copy(), gf.c_icz.copy(), dn.copy(), A, b, H, C, cs, ns)
    assert rel_err(g_A.download(9 * nnz), A) <= 1e-9
    gf.close()
