"""Which density pass ran (needs an MI355X): the FP64 one with its cubics in
LDS takes the steps of large boxes with few solutes, once the neighbour skin's
masks are there; the first force evaluation scans all offsets without it."""
import pytest

import misa_eam as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,cells,ratio,first,step", [
    (M.PREC_FP64, (64, 64, 64), (985, 10, 5), "kRhoDf", "kRhoDL"),
    (M.PREC_FP64, (64, 64, 64), (75, 15, 10), "kRhoDf", "kRhoDf"),
    (M.PREC_FP64, (12, 12, 12), (985, 10, 5), "kRhoDf", "kRhoDf"),
    (M.PREC_MIXED_KAHAN, (64, 64, 64), (985, 10, 5), "kRhoDfM", "kRhoDfM"),
])
def test_density_pass_used(setfl_fecuni, precision, cells, ratio, first, step):
    dev = M.EamDevice(cells)
    assert dev.density_pass() == "none"
    dev.make_offsets()
    dev.set_potential(setfl_fecuni)
    dev.set_precision(precision)
    dev.set_timestep(0.001)
    dev.build_world(5, 300.0, ratio, 5)
    dev.compute_forces()
    assert dev.density_pass() == first
    dev.step(2)
    assert dev.density_pass() == step
    dev.close()
