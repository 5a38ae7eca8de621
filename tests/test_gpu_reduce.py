"""The value reduction where blocks have unusual numbers of contributions -- all long, around the
length from which several lanes share a block, one or two, more than a workgroup stages at once -- in
every launch shape and added up as well as overwritten, and the CZ law at whole and other exponents
with masses of two and of more values, against the oracle."""
import numpy as np
import pytest

from conftest import rel_err
from icflow_amd import _lib
from workloads import H, Pipeline, make_state, small_specimen

pytestmark = pytest.mark.gpu

SHAPES = (None, (64, 2), (128, 3), (512, 2))


@pytest.mark.parametrize("precision", [_lib.ICF_FP64, _lib.ICF_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("alpha,beta,masses", [(4.0, 4.0, 2), (2.0, 16.0, 2), (3.7, 2.5, 2), (3.0, 17.0, 4)])
def test_blocks_of_any_length(orc, precision, alpha, beta, masses):
    bar = 1e-9 if precision == _lib.ICF_FP64 else 1e-5          # the parity bars of the two modes
    consts = _lib.consts_from_prms(**dict(_lib.SPECIMEN_PRMS, alpha=alpha, beta=beta))
    if masses == 4:
        m4 = np.array([[5, 1, 2, 3], [1, 6, 2, 1], [2, 2, 7, 1], [3, 1, 1, 8]], float) * consts.M[0] / 6
        consts.M[:] = np.kron(m4, np.eye(3)).ravel().tolist()
    col = small_specimen(cells=(5, 4, 4), size=(0.05, 0.04, 0.04), grains=6, seed=8, platens=False)
    p = Pipeline(col, consts, make_state(col, consts, seed=9), precision=precision)
    gf, lib, ctx = p.gf, p.gf.lib, p.gf.ctx
    T, C, N = len(col.elastic), len(col.czs), gf.csr.N
    es, cs, ns = gf.el_elastic_stride, gf.cz_stride, gf.nd_stride
    total = int((gf.c_ie_pcsr[4 * es:20 * es] >= 0).sum() + (gf.c_icz[10 * cs:46 * cs] >= 0).sum())
    orc.set_constants(consts)
    # contributions may cancel where many meet in a block: errors are measured against the largest of
    # the blocks' norm and that of the specimen's own blocks
    own, b = np.zeros(9 * gf.csr.nnz), np.zeros(3 * N)
    orc.elem_force(gf.c_ie_pcsr.copy(), gf.c_dn.copy(), H, own, b, T, es, ns)
    orc.cz_force(gf.c_dcz.copy(), gf.c_icz.copy(), gf.c_dn.copy(), own, b, H, C, cs, ns)
    rng = np.random.default_rng(10)
    g_b = gf.buf("b", 3 * N, np.float64)
    for nkeys in (1, 3, 65, 300, total // 9, total // 2):
        ie, icz = gf.c_ie_pcsr.copy(), gf.c_icz.copy()
        # most contributions at random, a run of blocks with exactly 8 and 9, the rest of the slots as they are
        to = np.concatenate([np.repeat(np.arange(min(nkeys, 60)), 8 + np.arange(min(nkeys, 60)) % 2)[:total // 3],
                             rng.integers(min(nkeys - 1, 60), nkeys, total)])[:total]
        to = rng.permutation(to)
        at = 0
        for a, lo, hi in ((ie, 4 * es, 20 * es), (icz, 10 * cs, 46 * cs)):
            on = np.nonzero(a[lo:hi] >= 0)[0] + lo
            a[on] = to[at:at + len(on)]
            at += len(on)
        A, b = np.zeros(9 * nkeys), np.zeros(3 * N)
        dn, dcz = gf.c_dn.copy(), gf.c_dcz.copy()
        orc.elem_force(ie.copy(), dn, H, A, b, T, es, ns)
        orc.cz_force(dcz, icz.copy(), dn, A, b, H, C, cs, ns)
        g_A = gf.buf("A", 9 * nkeys, np.float64)
        gf.g_ie_pcsr.upload(ie)
        first = None
        for shape in SHAPES:
            if shape:
                for acc in (0, 1):
                    for fp64 in (0, 1):
                        gf.set_chunk_keys(acc, fp64, *shape)
            for call in ("fused", "separate"):
                for buf, a in ((gf.g_icz, icz), (gf.g_dcz, gf.c_dcz), (gf.g_dn, gf.c_dn)):
                    buf.upload(a)
                if call == "fused":
                    _lib.check(lib.icf_assemble_elems_and_czs(ctx, gf.g_ie_pcsr.p, T, es, gf.g_dcz.p, gf.g_icz.p, C, cs,
                                                              gf.g_dn.p, ns, H, g_A.p, nkeys, g_b.p, N, None, None),
                               ctx, call)
                else:
                    g_A.zero()
                    g_b.zero()
                    _lib.check(lib.icf_elem_force(ctx, gf.g_ie_pcsr.p, gf.g_dn.p, H, g_A.p, g_b.p, T, es, ns), ctx, call)
                    _lib.check(lib.icf_cz_force(ctx, gf.g_dcz.p, gf.g_icz.p, gf.g_dn.p, g_A.p, g_b.p, H, C, cs, ns), ctx,
                               call)
                got = g_A.download(9 * nkeys)
                err = np.linalg.norm(got - A) / max(np.linalg.norm(A), np.linalg.norm(own))
                assert err <= bar and rel_err(g_b.download(3 * N), b) <= 1e-9, (nkeys, shape, call)
                first = got if first is None else first
                assert np.array_equal(got, first), (nkeys, shape, call)
    gf.close()
