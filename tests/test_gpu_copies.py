"""Frames between host arrays and the device (needs an MI355X).

Arrays of 4 MB and more come back through pinned slots of 2 MB that several
host threads empty; smaller ones, and calls that find the slots in use, are
copied directly.  Either way every byte arrives: at sizes around the
limit and a slot's end, from arrays at odd addresses, and with several
handles copying at once from threads of their own.
"""
import threading

import numpy as np
import pytest

import misa_eam as M
import oracle_py as O

pytestmark = pytest.mark.gpu

A = 2.855
F = 5.6 / 2.855


def _frame(setfl, cells, seed):
    sim = O.Sim(cells, A, F, setfl)
    sim.build_world(seed, 300.0, (985, 10, 5), seed)
    return sim.atoms().copy()


def _round_trip(dev, atoms):
    dev.upload(atoms)
    back, _ = dev.download()
    want, got = M.sub_box_view(atoms, dev), M.sub_box_view(back, dev)
    for k in ("id", "type", "x", "v"):
        np.testing.assert_array_equal(got[k], want[k], err_msg=k)
    return back


def _shifted(atoms, by):
    raw = np.empty(atoms.nbytes + 64, dtype=np.uint8)
    view = raw[by:by + atoms.nbytes].view(atoms.dtype).reshape(atoms.shape)
    view[...] = atoms
    return view


# the doubled ghost-extended array: 104 bytes a slot, 2 (n0 + 2 g)(n1 + 2 g)(n2 + 2 g) slots
@pytest.mark.parametrize("cells", [(20, 20, 21), (21, 21, 21), (21, 21, 22), (24, 25, 23), (40, 41, 42)])
def test_frame_round_trips(setfl_fecuni, cells):
    atoms = _frame(setfl_fecuni, cells, 3)
    print("copies: %s, %.3f MB" % (cells, atoms.nbytes / 2.0**20), flush=True)
    dev = M.EamDevice(cells)
    dev.make_offsets()
    dev.set_potential(setfl_fecuni)
    first = _round_trip(dev, atoms)
    again = _round_trip(dev, _shifted(atoms, 8))
    assert first.tobytes() == again.tobytes()
    dev.close()


def test_threads_copy_at_once(setfl_fecuni):
    cells = [(24, 24, 24), (26, 25, 24), (12, 12, 12), (28, 24, 24)]
    frames = [_frame(setfl_fecuni, c, 5 + k) for k, c in enumerate(cells)]
    errors = []

    def work(k):
        try:
            for _ in range(4):  # a handle's life as well: the last one gives the slots back
                dev = M.EamDevice(cells[k])
                dev.make_offsets()
                dev.set_potential(setfl_fecuni)
                for _ in range(3):
                    _round_trip(dev, frames[k])
                dev.close()
        except BaseException as e:  # noqa: B902
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(cells))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
