"""A run of steps in one call, whose inner steps take the next step's
predictor with the resultants, against the same steps one call each, which
never do: the same bits, rebuild steps and contacts."""
import pytest

from rockable_amd import decks as D
from tests import kat_decks as K
from tests.test_gpu_parity import _dynamic_hull_deck, assert_bodies_equal, assert_interactions_equal

pytestmark = pytest.mark.gpu


def _deck(name, d):
    if name == "dynamic":
        return _dynamic_hull_deck(d), None
    if name == "driven":
        return K.driven_plate(str(d), ["Control _x_Vel_ 0 0.1", "Control _z_For_ 0 40.0", "Control _zrot_Vel_ 0 0.5"],
                              dt=1e-5)
    if name == "bonds":
        shapes, deck = D.bonded_clusters_deck(n_clusters=2, cluster_dims=(3, 3, 2), clearance=1e-5, strength_mean=20.0)
    elif name == "viscous":
        shapes, deck = D.hull_packing_deck(n_bodies=65, lattice=(5, 5, 3), vmax=10.0, gap_factor=1.01,
                                           interverlet_steps=20, size_range=(5.8e-3, 6e-3))
        deck.body_force = "ViscousFluid 1000.0"
    else:
        n = {"one": 1, "33": 33, "600": 600}[name]
        shapes, deck = D.hull_packing_deck(n_bodies=n, lattice=(10, 10, 6), vmax=10.0, gap_factor=1.01,
                                           interverlet_steps=20, size_range=(5.8e-3, 6e-3))
    return D.write_deck(str(d), shapes, deck), None


@pytest.mark.parametrize("record", [0, 1])
@pytest.mark.parametrize("name", ["one", "33", "600", "viscous", "driven", "dynamic", "bonds"])
def test_run_equals_single_steps(tmp_path, name, record):
    from rockable_amd.engine import Engine
    path, driving = _deck(name, tmp_path)
    a, b = Engine(path, driving=driving), Engine(path, driving=driving)
    for e in (a, b):
        e.set_option("record_geometry", record)
        e.update_nl()
    for n in (1, 2, 137, 260):
        a.step(n)
        for _ in range(n):
            b.step(1)
        assert_bodies_equal(a.bodies(), b.bodies())
        assert a.counts()["nl_updates"] == b.counts()["nl_updates"]
    assert_interactions_equal(a.interactions(), b.interactions(), fields=("dn", "fn", "ft", "mom", "damp", "stick"))
    assert_bodies_equal(a.bodies(), b.bodies())


def test_heavy_walls_under_the_guard(tmp_path):
    """A floor and walls with more slots than heavy_min, left alone by the steps
    that go on, under a displacement check that freezes the steps inside
    most batches: at every read-out their resultants are those of a run of
    single steps, and the rebuild steps are the same."""
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=(24, 20, 2), spacing_factor=2.002, seed=6, vmax=0.05, nl="linkCells")
    deck.gravity = (30.0, -20.0, -400.0)
    deck.interVerlet = 1e3
    deck.dynamic_update_nl = 1
    deck.disp_update_nl, deck.angle_update_nl = 5e-7, 57.0
    path = D.write_deck(str(tmp_path), shapes, deck)
    a, b = Engine(path), Engine(path)
    for e in (a, b):
        e.set_option("record_geometry", 0)
        e.set_option("heavy_min", 20)
        e.update_nl()
    for n in (1, 90, 161):
        a.step(n)
        for _ in range(n):
            b.step(1)
        assert a.counts()["nl_updates"] == b.counts()["nl_updates"]
        assert_bodies_equal(a.bodies(), b.bodies())
    assert a.counts()["nl_updates"] > 10
    assert abs(a.bodies()["force"][0, 2]) > 0.0
