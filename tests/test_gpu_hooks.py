"""The accelerator hooks' density and force sums against the oracle's lattice
loops (needs an MI355X): boxes whose sites do not fill the last wavefront,
boxes as small as they may be, and vacancies next to one another, whose
records lie in one place.  Bars as in the parity tests: rho 1e-12, forces
1e-12 of max(|f|, rms)."""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855


@pytest.mark.parametrize("vacant", [0.0, 0.2], ids=["full", "vacancies"])
@pytest.mark.parametrize("cells", [(4, 4, 4), (5, 7, 6), (9, 8, 7)])
def test_hooks_match_oracle(setfl_fecuni, cells, vacant):
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(13, 300.0, (80, 12, 8), 13)
    sb = sim.sub_box()
    rng = np.random.default_rng(13)
    sb["x"] = sb["x"] + rng.uniform(-0.1, 0.1, sb["x"].shape)
    sb["type"][rng.uniform(size=sb["type"].shape) < vacant] = -1
    print("hooks: %s, %d vacancies" % (cells, int((sb["type"] < 0).sum())), flush=True)
    sim.phase("exchange_atom_first")
    sim.phase("clear_force")
    aos = sim.atoms().copy()
    sim.phase("lat_rho")
    sim.phase("rho_reverse")
    dev = M.EamDevice(cells)
    dev.make_offsets()
    dev.set_potential(setfl_fecuni)
    dev.lat_rho(aos, sim.rc)
    want, got = sim.sub_box(), M.sub_box_view(aos, dev)
    live = want["type"] >= 0
    np.testing.assert_allclose(got["rho"][live], want["rho"][live], rtol=1e-12)
    sim.phase("lat_df")
    sim.phase("df_forward")
    aos = sim.atoms().copy()
    aos["f"] = 0.0
    sim.phase("lat_force")
    sim.phase("force_reverse")
    dev.lat_force(aos, sim.rc)
    f, g = sim.sub_box()["f"][live], M.sub_box_view(aos, dev)["f"][live]
    norm = np.maximum(np.linalg.norm(f, axis=1), np.sqrt(np.mean(np.sum(f * f, axis=1))))
    assert (np.linalg.norm(g - f, axis=1) / norm).max() < 1e-12
    dev.close()
