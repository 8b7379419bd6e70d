"""The decide in one workgroup and over a grid (needs an MI355X).

A box of at most 100 000 sites takes its decide in one workgroup while its
lists are short, as seen at the last look: at the start of a call and every
128 steps.  A call of many steps and as many calls of one step choose
differently while the lists grow past that mark, and must end on the same
bits; and a box with inter atoms must agree with the oracle.
"""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O
from inter_cases import crafted_inter_state, oracle_forces_with_inter

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855
FIELDS = ("id", "type", "x", "v", "f", "rho", "df")


def _device(setfl, cells, precision=M.PREC_FP64):
    dev = M.EamDevice(cells)
    dev.make_offsets()
    dev.set_potential(setfl)
    dev.set_precision(precision)
    dev.set_timestep(0.001)
    return dev


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED_KAHAN], ids=["fp64", "mixed"])
@pytest.mark.parametrize("tset,pka", [(300.0, 2000.0), (1400.0, 0.0), (2600.0, 0.0)])
def test_one_call_equals_many(setfl_fecuni, tset, pka, precision):
    cells = (18, 17, 17)  # 10 404 sites
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(61, tset, (985, 10, 5), 61)
    atoms = sim.atoms().copy()
    devs = []
    for _ in range(2):
        dev = _device(setfl_fecuni, cells, precision)
        dev.upload(atoms)
        dev.compute_forces()
        if pka:
            dev.collision_step((9, 8, 8, 0), (1.0, 3.0, 5.0), pka)
        devs.append(dev)
    a, b = devs
    a.step(150)
    for _ in range(150):
        b.step(1)
    listed = a.defect_counters()
    print("decide forms: tset %g pka %g: %s" % (tset, pka, listed), flush=True)
    assert listed["staged"] > (0 if tset == 1400.0 else 64) and listed == b.defect_counters()
    (sa, ia), (sb, ib) = a.download(), b.download()
    va, vb = M.sub_box_view(sa, a), M.sub_box_view(sb, b)
    for k in FIELDS[:4]:
        np.testing.assert_array_equal(va[k], vb[k], err_msg=k)
        np.testing.assert_array_equal(ia[k], ib[k], err_msg="inter " + k)
    a.close()
    b.close()


@pytest.mark.parametrize("cells", [(17, 17, 17), (18, 17, 17)])  # 9 826 and 10 404 sites
def test_crafted_state_matches_oracle(setfl_fecuni, cells):
    """19 inter atoms, recombination and migration: ids, types and list order
    as the oracle's, positions to 1e-9 A as in the smaller boxes' test."""
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(23, 300.0, (985, 10, 5), 23)
    sb = sim.sub_box()
    sb["x"] = sb["x"] + np.random.default_rng(23).uniform(-0.08, 0.08, sb["x"].shape)
    inter = crafted_inter_state(sim, 23)
    dev = _device(setfl_fecuni, cells)
    dev.upload(sim.atoms().copy(), inter)
    dev.compute_forces()
    oracle_forces_with_inter(sim, inter)
    dev.step(10)
    sim.run(10)
    aos, got_inter = dev.download()
    got, want, wi = M.sub_box_view(aos, dev), sim.sub_box(), sim.inter()
    np.testing.assert_array_equal(got["type"], want["type"])
    live = want["type"] >= 0
    np.testing.assert_array_equal(got["id"][live], want["id"][live])
    np.testing.assert_array_equal(got_inter["id"], wi["id"])
    assert np.abs(got["x"] - want["x"]).max() < 1e-9
    if len(wi):
        assert np.abs(got_inter["x"] - wi["x"]).max() < 1e-9
    dev.close()
