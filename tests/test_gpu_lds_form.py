"""Which form of the force pass the automatic choice takes, and that the forms
agree (needs an MI355X).

The segments of like majority-species pairs are held in LDS.  The others go
through a queue while they are few; with many solutes, or a potential of so
many knots that those held begin beyond the nearest neighbours, the queue costs
more than masked gathers, and in the end the pass without LDS is the fastest.
The choice has to follow all of that, in single boxes and in batches, and the
form it takes ends on the bits of the pass without LDS.
"""
import numpy as np
import pytest

import misa_eam as M
import setfl_gen

pytestmark = pytest.mark.gpu

FIELDS = ("id", "type", "x", "v", "f", "rho", "df")
FE, DILUTE, RICH, MOST, NONE = (1, 0, 0), (985, 10, 5), (85, 10, 5), (40, 40, 20), (0, 60, 40)


@pytest.fixture(scope="module")
def potentials(tmp_path_factory):
    out = {}
    for nr in (5000, 10000, 20000):
        out[nr] = str(tmp_path_factory.mktemp("pot") / ("fecuni_%d.eam.alloy" % nr))
        setfl_gen.write_setfl(out[nr], ("Fe", "Cu", "Ni"), nr=nr)
    return out


def _box(pot, cells, ratio, precision, lds, tset=600.0, seed=5):
    dev = M.EamDevice(cells)
    dev.make_offsets()
    dev.set_potential(pot)
    dev.set_precision(precision)
    dev.set_lds_tables(lds)
    dev.set_timestep(0.001)
    dev.build_world(seed, tset, ratio, seed)
    dev.compute_forces()
    return dev


def _same(a, b, what):
    (sa, ia), (sb, ib) = a.download(), b.download()
    va, vb = M.sub_box_view(sa, a), M.sub_box_view(sb, b)
    for k in FIELDS:
        np.testing.assert_array_equal(va[k], vb[k], err_msg="%s: %s" % (what, k))
        np.testing.assert_array_equal(ia[k], ib[k], err_msg="%s: inter %s" % (what, k))


@pytest.mark.parametrize("precision,cells,ratio,nr,want", [
    (M.PREC_MIXED_KAHAN, (64, 63, 65), DILUTE, 5000, "kForceL"),
    (M.PREC_MIXED_KAHAN, (64, 63, 65), RICH, 5000, "kForceLG"),
    (M.PREC_MIXED_KAHAN, (64, 63, 65), FE, 10000, "kForceLG"),
    (M.PREC_MIXED, (64, 63, 65), DILUTE, 20000, "kForceLG"),
    (M.PREC_MIXED_F32SUM, (64, 63, 65), MOST, 5000, "kForceLG"),
    (M.PREC_MIXED_KAHAN, (64, 63, 65), NONE, 5000, "kForceM"),
    (M.PREC_MIXED_KAHAN, (40, 40, 40), DILUTE, 5000, "kForceM"),
    (M.PREC_FP64, (64, 63, 65), DILUTE, 5000, "kForceDL"),
    (M.PREC_FP64, (64, 63, 65), RICH, 5000, "kForceDG"),
    (M.PREC_FP64, (64, 63, 65), FE, 10000, "kForceDG"),
    (M.PREC_FP64, (64, 63, 65), MOST, 5000, "kForce"),
    (M.PREC_FP64, (64, 63, 65), MOST, 20000, "kForce"),
    (M.PREC_FP64, (40, 40, 40), DILUTE, 5000, "kForce"),
])
def test_automatic_form(potentials, precision, cells, ratio, nr, want):
    print("form: %s %s nr %d" % (cells, ratio, nr), flush=True)
    a, b = [_box(potentials[nr], cells, ratio, precision, m) for m in (M.LDS_AUTO, M.LDS_OFF)]
    assert a.force_pass() == want and b.force_pass() in ("kForce", "kForceM")
    _same(a, b, "first forces")
    a.step(3)
    b.step(3)
    assert a.force_pass() == want
    _same(a, b, "after 3 steps")
    a.close()
    b.close()


@pytest.mark.parametrize("precision,plain,lds", [(M.PREC_FP64, "kForce", "kForceDL"),
                                                 (M.PREC_MIXED_KAHAN, "kForceM", "kForceL")])
def test_boxes_about_as_large_as_the_persistent_launch(potentials, precision, plain, lds):
    """Sites that fill it a little more than once leave its second round empty."""
    for cells, want in (((50, 50, 50), plain), ((52, 51, 53), plain), ((56, 56, 56), lds)):
        dev = _box(potentials[5000], cells, DILUTE, precision, M.LDS_AUTO, 100.0)
        assert dev.force_pass() == want, cells
        dev.close()


@pytest.mark.parametrize("precision", [M.PREC_MIXED, M.PREC_MIXED_KAHAN, M.PREC_MIXED_F32SUM])
@pytest.mark.parametrize("ratio,nr", [(DILUTE, 5000), (MOST, 5000), (NONE, 5000), (FE, 20000)])
def test_batch_forms_end_on_the_bits_of_single_boxes(potentials, precision, ratio, nr):
    shapes = [(7, 6, 9), (12, 12, 12)]
    alone = [_box(potentials[nr], c, ratio, precision, M.LDS_OFF, 900.0, 7 + k) for k, c in enumerate(shapes)]
    boxes = [_box(potentials[nr], c, ratio, precision, M.LDS_AUTO, 900.0, 7 + k) for k, c in enumerate(shapes)]
    batch = M.EamBatch(boxes)
    for n in (5, 8):
        print("batch form: %s nr %d, %d steps" % (ratio, nr, n), flush=True)
        batch.step(n)
        for k, (a, b) in enumerate(zip(alone, boxes)):
            a.step(n)
            _same(a, b, "box %d after %d" % (k, n))
    batch.close()
    for d in alone + boxes:
        d.close()


def test_another_composition_takes_another_form(potentials):
    """An upload may turn a box from one form's to the other's."""
    cells = (64, 63, 65)
    dev = _box(potentials[5000], cells, DILUTE, M.PREC_MIXED_KAHAN, M.LDS_AUTO)
    ref = _box(potentials[5000], cells, RICH, M.PREC_MIXED_KAHAN, M.LDS_OFF)
    dev.step(2)
    assert dev.force_pass() == "kForceL"
    dev.build_world(5, 600.0, RICH, 5)
    dev.compute_forces()
    dev.step(2)
    ref.step(2)
    assert dev.force_pass() == "kForceLG"
    _same(dev, ref, "after the other upload")
    dev.close()
    ref.close()
