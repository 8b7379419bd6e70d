"""The forms of the lattice passes against one another and against the oracle
where they change over (needs an MI355X).

A box of few sites has four wavefronts to 64 sites, a larger one a wavefront
each, and the LDS passes walk the box in persistent blocks and work the pairs
with a solute off by whole wavefronts.  All of them sum the same terms in the
same order, so they end on the same bits: in the smallest boxes, where nearly
every site has ghost images on both sides, in odd ones, on either side of the
change from shared to single wavefronts, in boxes without the majority
species, and where so many atoms are far from their sites that every site
searches the whole neighbour list.
"""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855
FIELDS = ("id", "type", "x", "v", "f", "rho", "df")


def _device(setfl, cells, precision, lds, atoms):
    dev = M.EamDevice(cells)
    dev.make_offsets()
    dev.set_potential(setfl)
    dev.set_precision(precision)
    dev.set_lds_tables(lds)
    dev.upload(atoms)
    dev.set_timestep(0.001)
    dev.compute_forces()
    return dev


def _same(a, b, what):
    sa, ia = a.download()
    sb, ib = b.download()
    va, vb = M.sub_box_view(sa, a), M.sub_box_view(sb, b)
    for k in FIELDS:
        np.testing.assert_array_equal(va[k], vb[k], err_msg="%s: %s" % (what, k))
        np.testing.assert_array_equal(ia[k], ib[k], err_msg="%s: inter %s" % (what, k))


@pytest.mark.parametrize("precision", [M.PREC_MIXED_KAHAN, M.PREC_FP64], ids=["mixed", "fp64"])
@pytest.mark.parametrize("cells,ratio,tset", [
    ((4, 4, 4), (900, 70, 30), 1500.0),
    ((5, 7, 4), (0, 60, 40), 1500.0),
    ((9, 6, 11), (400, 300, 300), 1500.0),
    ((16, 17, 15), (1, 0, 0), 1500.0),
    ((40, 40, 80), (985, 10, 5), 300.0),   # the largest with four wavefronts to 64 sites
    ((40, 40, 84), (985, 10, 5), 300.0),   # just beyond
])
def test_force_forms_agree(setfl_fecuni, cells, ratio, tset, precision):
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(51, tset, ratio, 51)
    atoms = sim.atoms().copy()
    a, b = [_device(setfl_fecuni, cells, precision, m, atoms) for m in (M.LDS_OFF, M.LDS_ON)]
    _same(a, b, "first forces")
    for n in (1, 40):
        print("forms: %s, %d steps" % (cells, n), flush=True)
        a.step(n)
        b.step(n)
        _same(a, b, "after %d steps" % n)
    a.close()
    b.close()


@pytest.mark.parametrize("lds", [M.LDS_OFF, M.LDS_ON], ids=["shared", "lds"])
@pytest.mark.parametrize("cells", [(4, 4, 4), (5, 7, 6), (9, 8, 7)])
def test_far_atoms_everywhere_match_oracle(setfl_fecuni, cells, lds):
    """One atom in eight or more beyond 0.2a of its site: kWide on every site.
    FP64 bars as everywhere: rho 1e-12, forces 1e-12 of max(|f|, rms).  F' is
    compared through the forces: it passes through zero in this range of rho
    (-2e-5 next to -7e-2), where a relative bar says nothing about it."""
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(7, 300.0, (900, 70, 30), 7)
    sb = sim.sub_box()
    rng = np.random.default_rng(7)
    d = rng.normal(size=sb["x"].shape)
    d *= rng.uniform(0.5, 0.64, d.shape[:-1] + (1,)) / np.linalg.norm(d, axis=-1, keepdims=True)
    pick = rng.uniform(size=d.shape[:-1]) < 0.3
    sb["x"] = sb["x"] + d * pick[..., None]
    dev = _device(setfl_fecuni, cells, M.PREC_FP64, lds, sim.atoms().copy())
    sim.prepare()
    aos, _ = dev.download()
    got, want = M.sub_box_view(aos, dev), sim.sub_box()
    np.testing.assert_allclose(got["rho"], want["rho"], rtol=1e-12)
    f, g = want["f"].reshape(-1, 3), got["f"].reshape(-1, 3)
    norm = np.maximum(np.linalg.norm(f, axis=1), np.sqrt(np.mean(np.sum(f * f, axis=1))))
    assert (np.linalg.norm(g - f, axis=1) / norm).max() < 1e-12
    dev.close()
