"""What the accelerator hooks read and what they leave alone (needs an MI355X).

The force hook takes F' of a neighbour from the caller's FP64 record with all
its bits, whatever the neighbour's species; and a hook called between steps
leaves the resident state as it is, although it uses records of it as scratch.
"""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855
FIELDS = ("id", "type", "x", "v", "f", "rho", "df")


def _pair_force(dev, sim, kinds, df):
    """Force on an atom of kinds[0] with F' 0 from one of kinds[1] with F' df, all other sites vacant."""
    aos = sim.atoms().copy()
    aos["type"] = -1
    aos["f"] = 0.0
    aos["df"] = 0.0
    v = M.sub_box_view(aos, dev)  # [z, y, doubled x]
    v["type"][1, 1, 2], v["type"][1, 1, 3] = kinds
    v["df"][1, 1, 3] = df
    dev.lat_force(aos, sim.rc)
    return M.sub_box_view(aos, dev)["f"][1, 1, 2].copy()


@pytest.mark.parametrize("kinds", [(0, 0), (0, 1), (0, 2), (2, 1)])
def test_force_hook_takes_f_prime_whole(setfl_fecuni, kinds):
    cells = (4, 4, 4)
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(3, 0.0, (80, 12, 8), 3)
    sim.phase("exchange_atom_first")
    dev = M.EamDevice(cells)
    dev.make_offsets()
    dev.set_potential(setfl_fecuni)
    for base in (1.0e9, -3.0e7, 8.0):
        bits = np.float64(base).view(np.uint64)
        assert bits & np.uint64(3) == 0
        low = _pair_force(dev, sim, kinds, base)
        high = _pair_force(dev, sim, kinds, (bits | np.uint64(3)).view(np.float64))
        assert np.isfinite(low).all() and (low != 0).all()
        if abs(base) > 1.0e6:
            # the pair term is below 1e-3 of F' rho': three more units in the
            # last place of F' cannot be lost in the few roundings after it
            assert (np.abs(high) > np.abs(low)).all(), (kinds, base, low, high)
    for inf in (np.inf, -np.inf):
        f = _pair_force(dev, sim, kinds, inf)
        assert np.isinf(f).all(), (kinds, f)
        assert (np.sign(f) == np.sign(_pair_force(dev, sim, kinds, np.sign(inf) * 1.0e9))).all()
    dev.close()


@pytest.mark.parametrize("precision", [M.PREC_FP64, M.PREC_MIXED_KAHAN], ids=["fp64", "mixed"])
def test_steps_go_on_after_a_hook(setfl_fecuni, precision):
    cells = (7, 6, 8)
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(19, 900.0, (80, 12, 8), 19)
    sb = sim.sub_box()
    rng = np.random.default_rng(19)
    sb["type"][rng.uniform(size=sb["type"].shape) < 0.03] = -1
    atoms = sim.atoms().copy()
    sim.phase("exchange_atom_first")
    hooked = sim.atoms().copy()
    hooked["x"] += rng.uniform(-0.3, 0.3, hooked["x"].shape)  # another configuration than the resident one
    devs = []
    for _ in range(2):
        dev = M.EamDevice(cells)
        dev.make_offsets()
        dev.set_potential(setfl_fecuni)
        dev.set_precision(precision)
        dev.upload(atoms)
        dev.set_timestep(0.001)
        dev.compute_forces()
        devs.append(dev)
    plain, hook = devs
    for n in (1, 4, 3):
        plain.step(n)
        hook.lat_rho(hooked.copy(), sim.rc)
        hook.step(n)
        aos = hooked.copy()
        hook.lat_df(aos, sim.rc)
        hook.lat_force(aos, sim.rc)
    (sa, ia), (sh, ih) = plain.download(), hook.download()
    va, vh = M.sub_box_view(sa, plain), M.sub_box_view(sh, hook)
    for k in FIELDS:
        np.testing.assert_array_equal(va[k], vh[k], err_msg=k)
        np.testing.assert_array_equal(ia[k], ih[k], err_msg="inter " + k)
    for d in devs:
        d.close()
