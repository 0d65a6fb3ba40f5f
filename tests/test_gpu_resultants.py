"""The resultant kernel's slot windows, term passes and body groups: per-body
sums taken by it alone, at any slot count, equal the serial sums of the
heavy-body kernel bit for bit."""
import pytest

from tests.test_gpu_parity import assert_bodies_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 5, 4), (33, 31, 2), (70, 70, 2)])
@pytest.mark.parametrize("heavy_min", [10 ** 9, 64])
def test_slot_windows_match_serial_sums(tmp_path, dims, heavy_min):
    """A layer or two of spheres pressed on a floor: from one body, one past
    a group of 32, to a floor whose 4 900 contacts take two scan windows of
    4 096 slots and ten term passes of 512 (heavy_min 10^9: by the resultant
    kernel), against the serial sums of k_gather_heavy (heavy_min 8,
    exact_sums).  Same order of additions, so the bits are equal."""
    from rockable_amd import decks as D
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=dims, spacing_factor=2.002, seed=3, vmax=0.02, nl="linkCells")
    deck.gravity = (3.0, -2.0, -400.0)
    path = D.write_deck(str(tmp_path), shapes, deck)
    a, b = Engine(path), Engine(path)
    a.set_option("heavy_min", heavy_min)
    b.set_option("heavy_min", 8)
    for e in (a, b):
        e.set_option("exact_sums", 1)
        e.set_option("record_geometry", 0)
        e.update_nl()
        e.step(250)
    n = int(dims[0] * dims[1])
    assert a.counts()["nactive"] > n // 2
    assert_bodies_equal(a.bodies(), b.bodies())


@pytest.mark.parametrize("dims", [(180, 180, 1), (200, 170, 1)])
def test_threads_per_group_match_serial_sums(tmp_path, dims):
    """Floors on either side of the 1 024 groups of 32 bodies at which a group
    takes 128 threads instead of 256, against the serial sums of k_gather_heavy
    (heavy_min 1): bit for bit."""
    from rockable_amd import decks as D
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=dims, spacing_factor=2.002, seed=4, vmax=0.02, nl="linkCells")
    deck.gravity = (3.0, -2.0, -400.0)
    path = D.write_deck(str(tmp_path), shapes, deck)
    a, b = Engine(path), Engine(path)
    b.set_option("heavy_min", 1)
    for e in (a, b):
        e.set_option("exact_sums", 1)
        e.set_option("record_geometry", 0)
        e.update_nl()
        e.step(250)
    assert a.counts()["nactive"] > dims[0] * dims[1] // 2
    assert_bodies_equal(a.bodies(), b.bodies())
