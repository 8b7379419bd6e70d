"""The decide's early end: steps whose staged atoms all go straight back to
their sites, so that no list work is left (needs an MI355X).

The workgroup that does the list work ends early there.  Its first thread
clears the counters that the test for it looks at, so every wavefront has to
decide from what was read before: a wavefront that read them for itself could
see them half cleared and wait at barriers of its own.  The same steps are
taken in one workgroup (a single box) and over a grid (a batch), many at a
time, and must end on the same bits, where the oracle ends.
"""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855
FIELDS = ("id", "type", "x", "v", "f")


@pytest.mark.parametrize("cells", [(5, 5, 5), (9, 8, 7)])
@pytest.mark.parametrize("staged", [1, 16])
def test_steps_whose_staged_atoms_all_go_back(setfl_fecuni, cells, staged):
    steps = 11
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(31, 100.0, (985, 10, 5), 31)
    sb = sim.sub_box()
    flat = sb["x"].reshape(-1, 3)
    picked = np.random.default_rng(31).choice(len(flat), staged, replace=False)
    flat[picked, 0] += 0.72  # beyond 0.2 a, well within the site's own cell, and slow to return
    sb["x"] = flat.reshape(sb["x"].shape)
    devs = []
    for _ in range(2):
        dev = M.EamDevice(cells)
        dev.make_offsets()
        dev.set_potential(setfl_fecuni)
        dev.upload(sim.atoms().copy())
        dev.set_timestep(0.0005)
        dev.compute_forces()
        devs.append(dev)
    one, grid = devs
    one.step(steps)
    assert one.decide_forms() == (steps, 0)
    batch = M.EamBatch([grid])
    batch.step(steps)
    counts = one.defect_counters()
    print("decide exit: %s, %d displaced: %s" % (cells, staged, counts), flush=True)
    assert counts == grid.defect_counters()
    assert counts["staged"] == counts["refilled"] >= 2 * staged
    (sa, ia), (sb_, ib) = one.download(), grid.download()
    assert len(ia) == 0 and len(ib) == 0
    va, vb = M.sub_box_view(sa, one), M.sub_box_view(sb_, grid)
    for k in FIELDS:
        np.testing.assert_array_equal(va[k], vb[k], err_msg=k)
    sim.set_dt(0.0005)
    sim.prepare()
    sim.run(steps)
    want = sim.sub_box()
    np.testing.assert_array_equal(va["type"], want["type"])
    np.testing.assert_array_equal(va["id"], want["id"])
    assert np.abs(va["x"] - want["x"]).max() < 1e-9
    batch.close()
    one.close()
    grid.close()
