"""icf_pack_pcsr where slots already hold something: right values are kept, anything else --
other blocks of the same row, blocks of other rows, values outside the pattern -- is replaced,
and the assembly that follows uses the fields as they now are."""
import ctypes

import numpy as np
import pytest

from icflow_amd import _lib
from workloads import Pipeline, make_state, small_specimen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,grains", [((2, 2, 2), 2), ((3, 2, 5), 3), ((6, 5, 4), 6)])
@pytest.mark.parametrize("share", [0.0, 0.02, 1.0])
def test_pack_over_fields_in_any_state(specimen_consts, cells, grains, share):
    col = small_specimen(cells=cells, size=tuple(0.01 * c for c in cells), grains=grains, seed=3, platens=False)
    st = make_state(col, specimen_consts, seed=4)
    p = Pipeline(col, specimen_consts, st)
    gf, lib, ctx = p.gf, p.gf.lib, p.gf.ctx
    first = p.assemble()
    T, C, N, nnz = len(col.elastic), len(col.czs), gf.csr.N, gf.csr.nnz
    es, cs = gf.el_elastic_stride, gf.cz_stride
    alt = np.ascontiguousarray(col.alt, np.int32)

    def dev(name, a):
        b = gf.buf(name, a.size, a.dtype)
        b.upload(a)
        return b

    d_alt, d_rows, d_cols = dev("alt", alt), dev("p_rows", gf.csr.rows), dev("p_cols", gf.csr.cols)
    rng = np.random.default_rng(5)
    bad = np.array([-7, -1, 0, nnz - 1, nnz, 2 ** 31 - 1, -2 ** 31], np.int64)
    for host, buf, lo, hi in ((gf.c_ie_pcsr, gf.g_ie_pcsr, 4 * es, 24 * es), (gf.c_icz, gf.g_icz, 10 * cs, 52 * cs)):
        a = host.astype(np.int64)
        hit = rng.random(hi - lo) < share
        near = a[lo:hi] + rng.integers(-2, 3, hi - lo)
        a[lo:hi] = np.where(hit, np.where(rng.random(hi - lo) < 0.5, rng.choice(bad, hi - lo), near), a[lo:hi])
        buf.upload(a.astype(np.int32))
    for _ in range(2):                       # the second time nothing differs
        _lib.check(lib.icf_pack_pcsr(ctx, d_alt.p, len(alt), d_rows.p, d_cols.p, N, gf.g_ie_pcsr.p, T, es,
                                     gf.g_icz.p, C, cs, None, 0, 0), ctx, "pack_pcsr")
        got, want = gf.g_ie_pcsr.download().reshape(-1, es), gf.c_ie_pcsr.reshape(-1, es)
        assert np.array_equal(got[:24, :T], want[:24, :T])
        got, want = gf.g_icz.download().reshape(-1, cs), gf.c_icz.reshape(-1, cs)
        assert np.array_equal(got[4:52, :C], want[4:52, :C])
        gf.TransferNodesToGPU(st)
        gf.g_dcz.upload(gf.c_dcz)
        again = p.assemble()
        for k in ("vals", "rhs", "F", "dcz"):
            assert np.array_equal(first[k], again[k]), k
    gf.close()


def test_changed_slots_reach_the_assembly(specimen_consts):
    """A second pattern packed into the same buffers between two assemblies, and back."""
    col = small_specimen(cells=(5, 4, 4), size=(0.05, 0.04, 0.04), grains=5, seed=9)
    st = make_state(col, specimen_consts, seed=10, platen_dz_frac=0.3)
    p = Pipeline(col, specimen_consts, st, contact=True)
    gf, lib, ctx = p.gf, p.gf.lib, p.gf.ctx
    T, C, N = len(col.elastic), len(col.czs), gf.csr.N
    es, cs = gf.el_elastic_stride, gf.cz_stride
    alt = np.ascontiguousarray(col.alt, np.int32)
    wide = (gf.csr.rows.copy(), gf.csr.cols.copy())     # with the impacts' blocks
    gf.CreateStructure(None)
    plain = (gf.csr.rows.copy(), gf.csr.cols.copy())
    assert len(wide[1]) > len(plain[1])
    d_alt = gf.buf("alt", alt.size, np.int32)
    d_alt.upload(alt)
    d_rows, d_cols = gf.buf("p_rows", N + 1, np.int32), gf.buf("p_cols", len(wide[1]), np.int32)
    g_vals, g_rhs = gf.buf("v", 9 * len(wide[1]), np.float64), gf.buf("r", 3 * N, np.float64)
    dense = []
    for rows, cols in (plain, wide, plain):
        d_rows.upload(rows)
        d_cols.upload(cols)
        _lib.check(lib.icf_pack_pcsr(ctx, d_alt.p, len(alt), d_rows.p, d_cols.p, N, gf.g_ie_pcsr.p, T, es, gf.g_icz.p,
                                     C, cs, None, 0, 0), ctx, "pack_pcsr")
        _lib.check(lib.icf_assemble_elems_and_czs(ctx, gf.g_ie_pcsr.p, T, es, gf.g_dcz.p, gf.g_icz.p, C, cs, gf.g_dn.p,
                                                  gf.nd_stride, 1e-4, g_vals.p, len(cols), g_rhs.p, N, None, None),
                   ctx, "assemble")
        v = g_vals.download(9 * len(cols)).reshape(-1, 9)
        r = np.repeat(np.arange(N), np.diff(rows))
        dense.append({(a, b): x for a, b, x in zip(r.tolist(), cols.tolist(), v)})
    assert dense[0].keys() == dense[2].keys()
    for key, x in dense[1].items():
        want = dense[0].get(key, np.zeros(9))
        assert np.array_equal(x, want), key
        assert key not in dense[2] or np.array_equal(dense[2][key], want), key
    gf.close()
