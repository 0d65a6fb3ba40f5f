"""Read-outs packed on the device: the active interactions against the listed
ones filtered on the host, with the counts and a cap, and the bodies against a
saved deck, over counts around the packing's blocks."""
import ctypes

import numpy as np
import pytest

from rockable_amd import decks as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (6, 6, 5), (12, 11, 9)])
def test_active_records_and_counts(tmp_path, dims):
    from rockable_amd.engine import INTERACTION_DTYPE, Engine
    shapes, deck = D.sphere_lattice_deck(dims=dims, spacing_factor=2.002, seed=5, vmax=0.05, nl="linkCells")
    deck.gravity = (5.0, 3.0, -300.0)
    e = Engine(D.write_deck(str(tmp_path), shapes, deck))
    e.update_nl()
    for steps in (0, 1, 150, 151):
        e.step(steps)
        every = e.interactions()
        act = e.interactions(active=True)
        want = every[(every["dn"] < 0) | (every["stick"] >= 0)]
        assert e.counts()["nlisted"] == len(every)
        if steps:  # (before the first step the list is new and nothing is active)
            assert e.counts()["nactive"] == len(act) == len(want)
            assert act.tobytes() == want.tobytes()
        cap = len(act) // 2
        part = np.zeros(cap + 1, dtype=INTERACTION_DTYPE)
        n = ctypes.c_size_t(0)
        assert e.L.rk_get_interactions(e.h, 1, part.ctypes.data, cap, ctypes.byref(n)) == 0
        assert n.value == len(act) and part[:cap].tobytes() == act[:cap].tobytes()
        assert not np.any(part[cap:].view(np.uint8))
    e.save_conf(str(tmp_path / "out.conf"))
    _, saved = D.read_conf_bodies(str(tmp_path / "out.conf"))
    b = e.bodies()
    for k in ("pos", "Q", "vel", "vrot", "acc", "arot"):
        assert np.allclose(b[k], saved[k], rtol=1e-14, atol=1e-300)
