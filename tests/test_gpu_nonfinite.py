"""A lattice atom without a finite position, or too far out for an FP32
displacement, is within no other atom's cutoff (needs an MI355X).

In FP64 and in the mixed modes with FP64 or plain FP32 sums such an atom counts
for none of its neighbours: their densities and forces are those of a box where
its site is vacant, bit for bit, in every form of the passes, and the call
succeeds.  (With compensated sums it fails the call.)
"""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855


@pytest.mark.parametrize("lds", [M.LDS_ON, M.LDS_OFF], ids=["lds", "global"])
@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED, M.PREC_MIXED_F32SUM])
@pytest.mark.parametrize("where", [np.nan, np.inf, -np.inf, 1.0e39])
def test_atom_out_of_every_cutoff(setfl_fecuni, where, precision, lds):
    cells = (8, 7, 6)
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(3, 300.0, (80, 12, 8), 3)
    sb = sim.sub_box()
    sb["x"] = sb["x"] + np.random.default_rng(3).uniform(-0.1, 0.1, sb["x"].shape)
    got = []
    for vacant in (False, True):
        aos = sim.atoms().copy()
        dev = M.EamDevice(cells)
        dev.make_offsets()
        dev.set_potential(setfl_fecuni)
        dev.set_precision(precision)
        dev.set_lds_tables(lds)
        v = M.sub_box_view(aos, dev)
        for site in ((3, 3, 6), (3, 3, 7), (0, 0, 0)):  # two next to one another, one at the corner
            if vacant:
                v["type"][site] = -1
            else:
                v["x"][site][1] = where
        dev.upload(aos)
        dev.compute_forces()
        out, _ = dev.download()
        got.append(M.sub_box_view(out, dev).copy())
        dev.close()
    live = got[1]["type"] >= 0
    assert np.isfinite(got[0]["f"]).all()
    for k in ("rho", "df", "f"):
        np.testing.assert_array_equal(got[0][k][live], got[1][k][live], err_msg=k)
    # in FP64 two atoms side by side at 1e39 A are at a distance of each other like any two
    if precision != M.PREC_FP64 or not np.isfinite(where):
        assert (got[0]["f"][~live] == 0).all()
