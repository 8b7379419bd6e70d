"""Boxes with more inter atoms than the wavefronts that work them off (needs an
MI355X): the site passes carry the inter atoms in their first blocks, the LDS
passes spread them over all of theirs.  Either way one wavefront sums one atom
at a time in a fixed order, so both end on the same bits."""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855
FIELDS = ("id", "type", "x", "v", "f", "rho", "df")


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED_KAHAN], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n_inter", [1, 1023, 1025, 2500])
def test_many_inter_atoms(setfl_fecuni, n_inter, precision):
    n = 18
    sim = O.Sim((n, n, n), A, F, setfl_fecuni)
    sim.build_world(3, 50.0, (900, 70, 30), 3)
    atoms = sim.atoms().copy()
    c = np.random.default_rng(n_inter).choice(n ** 3, n_inter, replace=False)
    inter = np.zeros(n_inter, dtype=O.ATOM_DTYPE)
    inter["id"] = 10 ** 7 + np.arange(n_inter)
    inter["type"] = np.arange(n_inter) % 3
    inter["x"] = np.stack([c % n + 0.5, c // n % n + 0.5, c // n // n + 0.004], 1) * A  # face centres
    print("inter atoms: %d" % n_inter, flush=True)
    devs = []
    for lds in (M.LDS_OFF, M.LDS_ON):
        dev = M.EamDevice((n, n, n))
        dev.make_offsets()
        dev.set_potential(setfl_fecuni)
        dev.set_precision(precision)
        dev.set_lds_tables(lds)
        dev.set_timestep(1.0e-5)
        dev.upload(atoms, inter)
        dev.compute_forces()
        dev.step(4)
        devs.append(dev)
    (sa, ia), (sb, ib) = [d.download() for d in devs]
    assert len(ia) == len(ib) == n_inter
    va, vb = M.sub_box_view(sa, devs[0]), M.sub_box_view(sb, devs[1])
    assert np.isfinite(ia["f"]).all() and (ia["rho"] > 0).all()
    for k in FIELDS:
        np.testing.assert_array_equal(va[k], vb[k], err_msg=k)
        np.testing.assert_array_equal(ia[k], ib[k], err_msg="inter " + k)
    for d in devs:
        d.close()
