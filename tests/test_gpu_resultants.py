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


def _glued_bed(d, dims, ndriven, dynamic=False, body_force=None):
    """Layers of spheres pressed on each other, the first ndriven of the lowest
    one and the walls driven; controls on four of the grains."""
    from rockable_amd import decks as D
    shapes, deck = D.sphere_lattice_deck(dims=dims, spacing_factor=2.002, seed=8, vmax=0.05, nl="linkCells")
    walls, grains = deck.bodies[:5], deck.bodies[5:]
    low = [b for k, b in enumerate(grains) if k % dims[2] == 0]
    for b in low[:ndriven - 5]:
        b.vel = (0.0, 0.0, 0.0)
    deck.bodies = walls + low + [b for k, b in enumerate(grains) if k % dims[2]]
    deck.nDriven = ndriven
    deck.gravity = (30.0, -20.0, -400.0)
    deck.body_force = body_force
    if dynamic:
        deck.interVerlet = 1e3
        deck.dynamic_update_nl = 1
        deck.disp_update_nl, deck.angle_update_nl = 1e-6, 57.0
    path = D.write_deck(str(d), shapes, deck)
    drv = str(d / "drivingSystem.txt")
    with open(drv, "w") as fh:
        fh.write("Control _z_Vel_ 5 0.02\nControl _x_Vel_ %d -0.03\nControl _z_For_ 700 1e-3\nControl _zrot_Mom_ 701 1e-9\n"
                 % (ndriven - 1))
    return path, drv


@pytest.mark.parametrize("body_force", [None, "ViscousFluid 1000.0"])
@pytest.mark.parametrize("dims,ndriven", [((45, 46, 2), 2047), ((45, 46, 2), 2048), ((72, 72, 2), 5123)])
def test_many_driven_bodies_match_oracle(tmp_path, dims, ndriven, body_force):
    """Up to and past the 2 048 driven bodies from which a workgroup takes
    several (with a last group that is not full): sums, rebuilds and motion
    equal the serial oracle's."""
    from oracle.rk_oracle import Oracle
    from rockable_amd.engine import Engine
    path, drv = _glued_bed(tmp_path, dims, ndriven, body_force=body_force)
    e, o = Engine(path, driving=drv), Oracle(path, driving=drv, threads=8)
    e.set_option("record_geometry", 0)
    e.set_option("heavy_min", 10 ** 9)
    e.update_nl()
    o.update_nl()
    for n in (1, 250):
        e.step(n)
        o.run_steps(n)
        assert_bodies_equal(e.bodies(), o.bodies())
    assert e.counts()["nactive"] == o.nactive > ndriven // 3


@pytest.mark.parametrize("dynamic", [False, True])
def test_many_driven_bodies_with_heavy_ones(tmp_path, dynamic):
    """Groups of driven bodies that hold a heavy one, the floor first: its
    slots are left to the heavy kernels, the others' sums unchanged, under the
    displacement check too; against single steps and against a skip_far 0
    run."""
    from rockable_amd.engine import Engine
    path, drv = _glued_bed(tmp_path, (72, 72, 2), 5123, dynamic)
    engines = [Engine(path, driving=drv) for _ in range(3)]
    for k, e in enumerate(engines):
        e.set_option("record_geometry", 0)
        e.set_option("skip_far", 0 if k == 2 else 1)
        e.update_nl()
    a, b, c = engines
    for n in (1, 250):
        a.step(n)
        c.step(n)
        for _ in range(n):
            b.step(1)
        assert_bodies_equal(a.bodies(), b.bodies())
        assert_bodies_equal(a.bodies(), c.bodies())
        assert a.counts()["nl_updates"] == b.counts()["nl_updates"] == c.counts()["nl_updates"]
    assert a.counts()["nactive"] > 1000
    assert not dynamic or a.counts()["nl_updates"] > 2


@pytest.mark.parametrize("dims", [(60, 60, 1), (200, 170, 1), (363, 363, 1)])
def test_body_force_forms_match_serial_sums(tmp_path, dims):
    """The resultant kernel's forms with a body force: 256 threads to a group of
    32 bodies, 128, and 128 to a group of 64 from 131 072 bodies, against the
    serial sums of k_gather_heavy (heavy_min 1)."""
    from rockable_amd import decks as D
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=dims, spacing_factor=2.002, seed=4, vmax=0.05, nl="linkCells")
    deck.gravity = (3.0, -2.0, -400.0)
    deck.body_force = "ViscousFluid 1000.0"
    path = D.write_deck(str(tmp_path), shapes, deck)
    a, b = Engine(path), Engine(path)
    b.set_option("heavy_min", 1)
    for e in (a, b):
        e.set_option("exact_sums", 1)
        e.set_option("record_geometry", 0)
        e.update_nl()
        e.step(120)
    assert a.counts()["nactive"] > dims[0] * dims[1] // 8
    assert_bodies_equal(a.bodies(), b.bodies())
