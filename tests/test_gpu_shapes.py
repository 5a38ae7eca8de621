"""What an untuned context reports of its launch shapes (icf_get_autotune, icf_get_shape) is what its
launches use, and keeping it for a later run changes nothing there."""
import numpy as np
import pytest

from icflow_amd import _lib
from workloads import Pipeline, make_state, small_specimen

pytestmark = pytest.mark.gpu

BEFORE = {"phase1": 256, "narrow": 256, "closest": 8, "impact": 256, "order": 1}
# a few hundred tets and impacts: one-wave values, phase 1 and impacts with 64 lanes, forces first
AFTER = {"phase1": 64, "narrow": 256, "closest": 8, "impact": 64, "order": 0}


@pytest.mark.parametrize("precision", [_lib.ICF_FP64, _lib.ICF_MIXED], ids=["fp64", "mixed"])
def test_untuned_shapes_are_reported(specimen_consts, precision):
    col = small_specimen(cells=(5, 4, 4), size=(0.05, 0.04, 0.04), grains=5, seed=33)
    st = make_state(col, specimen_consts, seed=34, platen_dz_frac=0.3)
    stage, other = ("fp64", "fp32") if precision == _lib.ICF_FP64 else ("fp32", "fp64")
    default = [256, 3] if other == "fp64" else [256, 2]

    def run(shapes=None):
        p = Pipeline(col, specimen_consts, st, precision=precision, contact=True)
        assert len(p.impacts) > 0
        assert {r: v[0] for r, v in p.gf.shape_state().items()} == BEFORE
        if shapes:
            p.gf.use_shapes(shapes)
        return p, p.assemble()

    p, ref = run()
    kept = p.gf.tuned_shapes()
    for r, want in AFTER.items():
        assert kept[r] == want, (r, kept[r])
    assert kept["overwrite," + stage] == [64, 3] and kept["accumulate," + stage] == [128, 3]
    assert kept["overwrite," + other] == default and kept["accumulate," + other] == default   # never launched
    # in a context that keeps them, and in one that goes by itself again
    for shapes in (kept, None):
        q, got = run(shapes)
        assert q.gf.tuned_shapes() == kept
        for k in ("vals", "rhs", "F", "dcz"):
            assert np.array_equal(got[k], ref[k]), k
        q.gf.close()
    # stage 0 keeps the staging that is reported
    p.gf.set_chunk_keys(1, precision == _lib.ICF_FP64, 256, 0)
    assert p.gf.tuned_shapes()["accumulate," + stage] == [256, 3]
    # what is set is what is reported
    p.gf.set_shape("phase1", 128)
    p.gf.set_chunk_keys(0, precision == _lib.ICF_FP64, 512, 2)
    p.gf.g_dn.upload(np.zeros(3 * p.gf.nd_stride), offset_elems=12 * p.gf.nd_stride)
    p.assemble()
    kept = p.gf.tuned_shapes()
    assert kept["phase1"] == 128 and kept["overwrite," + stage] == [512, 2]
    p.gf.close()
