"""The sums of the pairs that the LDS force pass sets aside, mixed precision
(needs an MI355X): FP64 terms in offset order, whichever pass takes them.

With FP64 sums the force of a single pair is the exact FP64 product of its FP32
factor and the FP32 displacement: its components stand to one another as those
of the displacement, to FP64 rounding (2^-53 each side, one division: 1e-15).
A sum on any coarser grid misses that.  In an alloy with solutes on most sites,
where one site's pairs fill several full wavefronts of the queue, the pass with
the queue and those without it must agree bit for bit.
"""
import numpy as np
import pytest

import misa_eam as M
import oracle_py as O

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855


def _device(setfl, cells, precision, lds):
    dev = M.EamDevice(cells)
    dev.make_offsets()
    dev.set_potential(setfl)
    dev.set_precision(precision)
    dev.set_lds_tables(lds)
    return dev


@pytest.mark.parametrize("lds", [M.LDS_ON, M.LDS_OFF], ids=["queue", "inline"])
@pytest.mark.parametrize("kinds", [(0, 1), (1, 0), (1, 1), (2, 0)])
def test_force_of_one_pair_is_an_exact_product(setfl_fecuni, kinds, lds):
    cells = (8, 8, 8)
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(3, 0.0, (80, 12, 8), 3)
    dev = _device(setfl_fecuni, cells, M.PREC_MIXED, lds)
    aos = sim.atoms().copy()
    aos["type"] = -1
    v = M.sub_box_view(aos, dev)  # [z, y, doubled x]
    v["type"][3, 3, 6], v["type"][3, 3, 9] = kinds  # 1.5 a, 0.5 a, 0.5 a apart
    dev.upload(aos)
    dev.compute_forces()
    assert dev.force_pass() == ("kForceL" if lds == M.LDS_ON else "kForceM")
    out, _ = dev.download()
    d = np.array([1.5 * A, 0.5 * A, 0.5 * A]).astype(np.float32).astype(np.float64)
    for X in (6, 9):
        f = M.sub_box_view(out, dev)["f"][3, 3, X]
        print("set aside: %s X %d f %s" % (kinds, X, f), flush=True)
        assert (f != 0).all()
        assert np.abs(f / d / (f[0] / d[0]) - 1.0).max() < 1e-15
    dev.close()


@pytest.mark.parametrize("ratio", [(985, 10, 5), (40, 35, 25), (0, 60, 40)])
@pytest.mark.parametrize("precision", [M.PREC_MIXED, M.PREC_MIXED_KAHAN, M.PREC_MIXED_F32SUM])
def test_queue_gives_the_bits_of_the_other_passes(setfl_fecuni, precision, ratio):
    cells = (9, 8, 10)
    sim = O.Sim(cells, A, F, setfl_fecuni)
    sim.build_world(29, 600.0, ratio, 29)
    sb = sim.sub_box()
    rng = np.random.default_rng(29)
    sb["x"] = sb["x"] + rng.uniform(-0.2, 0.2, sb["x"].shape)
    sb["type"][rng.uniform(size=sb["type"].shape) < 0.02] = -1
    atoms = sim.atoms().copy()
    forces = []
    for lds in (M.LDS_ON, M.LDS_OFF, M.LDS_ON):
        dev = _device(setfl_fecuni, cells, precision, lds)
        dev.upload(atoms)
        dev.compute_forces()
        out, _ = dev.download()
        forces.append(M.sub_box_view(out, dev)["f"].copy())
        dev.close()
    assert np.isfinite(forces[0]).all()
    np.testing.assert_array_equal(forces[0], forces[1])
    np.testing.assert_array_equal(forces[0], forces[2])
