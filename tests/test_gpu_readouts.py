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


@pytest.mark.parametrize("n", [0, 1, 300, 20966, 20967])
def test_bodies_by_mapped_memory_and_by_copies(tmp_path, n):
    """All arrays at once, pairs and single ones, up to the 20 971 bodies read
    out through mapped host memory and one more, which goes by copies: the
    same bytes, and nothing written past the bodies."""
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=(28, 28, 27), spacing_factor=2.002, seed=5, vmax=0.05, nl="linkCells")
    deck.bodies = deck.bodies[:deck.nDriven + n]
    deck.gravity = (5.0, 3.0, -300.0)
    e = Engine(D.write_deck(str(tmp_path), shapes, deck))
    e.update_nl()
    e.step(60)
    names = ("pos", "Q", "vel", "vrot", "acc", "arot", "force", "moment")
    nb = deck.nDriven + n

    def read(want):
        out = [np.full((nb + 1, 4 if k == "Q" else 3), 7.25) for k in names]
        ptr = [a.ctypes.data if k in want else None for k, a in zip(names, out)]
        assert e.L.rk_get_bodies(e.h, *ptr, nb) == 0
        for k, a in zip(names, out):
            assert np.all(a[nb if k in want else 0:] == 7.25)
        return {k: a[:nb] for k, a in zip(names, out) if k in want}
    every = read(names)
    for want in [(k,) for k in names] + [("pos", "vel"), ("Q", "force"), ()]:
        part = read(want)
        for k in want:
            assert part[k].tobytes() == every[k].tobytes(), k
    e.save_conf(str(tmp_path / "out.conf"))
    _, saved = D.read_conf_bodies(str(tmp_path / "out.conf"))
    for k in ("pos", "Q", "vel", "vrot", "acc", "arot"):
        assert np.allclose(every[k], saved[k], rtol=1e-14, atol=1e-300)
    if n >= 300:
        assert np.abs(every["force"]).max() > 0.0


@pytest.mark.parametrize("dims", [(23, 23, 23), (29, 29, 29)])
def test_active_count_by_host_and_device(tmp_path, dims):
    """Lists shorter and longer than the 65 536 entries that the host counts."""
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=dims, spacing_factor=2.002, seed=5, vmax=0.05, nl="linkCells")
    e = Engine(D.write_deck(str(tmp_path), shapes, deck))
    e.update_nl()
    e.step(80)
    c = e.counts()
    assert (c["nlisted"] > 65536) == (dims[0] == 29)
    assert c["nactive"] == len(e.interactions(active=True)) == e.stats()["nactive"] > 100
