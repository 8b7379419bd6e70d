"""Both forms of the decide, seen to run, on the same states (needs an MI355X).

A box of at most 100 000 sites takes its decide in one workgroup while at most
32 entries (inter atoms, their images, far atoms) are listed at the last look,
and over a grid with more.  The library tells which ran.
"""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O
from inter_cases import crafted_inter_state, oracle_forces_with_inter

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855


def _device(setfl, cells, precision):
    dev = M.EamDevice(cells)
    dev.make_offsets()
    dev.set_potential(setfl)
    dev.set_precision(precision)
    dev.set_timestep(0.001)
    return dev


@pytest.mark.parametrize("n_inter,form", [(3, 0), (19, 1)], ids=["one-workgroup", "grid"])
def test_crafted_states_in_either_form(setfl_fecuni, n_inter, form):
    """Inter atoms, recombination and migration against the oracle: ids, types
    and list order, positions to 1e-9 A as in the smaller boxes' test."""
    cells = (13, 12, 11)
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(23, 300.0, (985, 10, 5), 23)
    sb = sim.sub_box()
    sb["x"] = sb["x"] + np.random.default_rng(23).uniform(-0.08, 0.08, sb["x"].shape)
    inter = crafted_inter_state(sim, 23)[:n_inter].copy()
    dev = _device(setfl_fecuni, cells, M.PREC_FP64)
    dev.upload(sim.atoms().copy(), inter)
    dev.compute_forces()
    oracle_forces_with_inter(sim, inter)
    used = np.zeros(2, dtype=np.int64)
    for _ in range(10):
        dev.step(1)
        used += dev.decide_forms()
    sim.run(10)
    print("decide forms used: %d inter atoms: %s" % (n_inter, used), flush=True)
    assert used[form] > 0
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


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED_KAHAN], ids=["fp64", "mixed"])
def test_lists_that_outgrow_one_workgroup(setfl_fecuni, precision):
    """One call stays in one workgroup for its first 128 steps, single steps
    change over as the cascade's lists grow: the same bits."""
    cells = (18, 17, 17)
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(61, 300.0, (985, 10, 5), 61)
    atoms = sim.atoms().copy()
    devs = []
    for _ in range(2):
        dev = _device(setfl_fecuni, cells, precision)
        dev.upload(atoms)
        dev.compute_forces()
        dev.collision_step((9, 8, 8, 0), (1.0, 3.0, 5.0), 2000.0)
        devs.append(dev)
    a, b = devs
    a.step(120)
    used = np.zeros(2, dtype=np.int64)
    for _ in range(120):
        b.step(1)
        used += b.decide_forms()
    print("decide forms used: one call %s, single steps %s" % (a.decide_forms(), used), flush=True)
    assert a.decide_forms() == (120, 0)
    assert used.sum() == 120 and used.min() > 0
    assert a.defect_counters() == b.defect_counters()
    (sa, ia), (sb, ib) = a.download(), b.download()
    va, vb = M.sub_box_view(sa, a), M.sub_box_view(sb, b)
    for k in ("id", "type", "x", "v"):
        np.testing.assert_array_equal(va[k], vb[k], err_msg=k)
        np.testing.assert_array_equal(ia[k], ib[k], err_msg="inter " + k)
    a.close()
    b.close()
