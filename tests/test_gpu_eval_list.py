"""The evaluation list of the steps that write no geometry records: counts
around its tiles of 1024 entries and its eight parts, faces of three, four
and more vertices, a flow whose motion is mostly common, against steps that
evaluate every entry (skip_far 0): same bits, gaps and rebuild steps."""
import numpy as np
import pytest

from rockable_amd import decks as D
from tests.test_gpu_parity import assert_bodies_equal, assert_interactions_equal

pytestmark = pytest.mark.gpu


def _prism(n, h, r):
    """A prism over a regular n-gon: two faces of n vertices."""
    a = 2 * np.pi * np.arange(n) / n
    v = np.array([(np.cos(x), np.sin(x), z) for z in (-0.5 * h, 0.5 * h) for x in a])
    edge = [(k, (k + 1) % n) for k in range(n)] + [(n + k, n + (k + 1) % n) for k in range(n)] + \
        [(k, n + k) for k in range(n)]
    face = [list(range(n)), list(range(n, 2 * n))] + [[k, (k + 1) % n, n + (k + 1) % n, n + k] for k in range(n)]
    return D.Shape("PRISM%d" % n, r, v, edge, face, volume=0.5 * n * np.sin(2 * np.pi / n) * h,
                   inertia_mass=(0.3, 0.3, 0.4))


@pytest.mark.parametrize("n,flow", [(1, 0.0), (30, 0.0), (200, 0.0), (200, 3.0), (700, -5.0)])
def test_list_equals_full_evaluation(tmp_path, n, flow):
    from rockable_amd.engine import Engine
    rng = np.random.default_rng(n)
    walls, wb = D.box_walls((-0.2, -0.03, 0.0), (0.4, 0.08, 0.2), 2e-4)
    pool = [_prism(k, 0.8, 0.05) for k in (3, 4, 5, 7)] + [D.sphere_shape("BALL", 0.6)]
    deck = D.Deck(dt=1e-6, tmax=1.0, interVerlet=3e-5, DVerlet=6e-4, dVerlet=3e-4, density={0: 2700.0, 1: 2700.0},
                  gravity=(20.0, 0.0, -90.0), update_nl="linkCells", nDriven=len(wb), force_law="Avalanche",
                  params=D.contact_params(1e6, 8e5, 0.25, 0.4, groups=((0, 0), (0, 1))))
    deck.cell_min_sizes = (0.012, 0.012, 0.012)
    deck.box_for_linkcells_opt = 1
    deck.bodies = list(wb)
    for k in range(n):
        p = (0.006 + 0.0097 * (k % 6), 0.006 + 0.0097 * (k // 6 % 5), 0.0046 + 0.0091 * (k // 30))
        v = rng.uniform(-1.0, 1.0, 3) + (flow, 0.0, -1.0)
        deck.bodies.append(D.Body(pool[k % len(pool)].name, homothety=0.0042, pos=p, vel=tuple(v),
                                  Q=tuple(D.small_rotations(rng, 1, 0.1)[0]), vrot=tuple(rng.uniform(-50, 50, 3))))
    path = D.write_deck(str(tmp_path), walls + pool, deck)
    a, b = Engine(path), Engine(path)
    for e, skip in ((a, 1), (b, 0)):
        e.set_option("record_geometry", 0)
        e.set_option("skip_far", skip)
        e.update_nl()
    contacts = 0
    for steps in (1, 40, 300, 400):
        a.step(steps)
        b.step(steps)
        assert_bodies_equal(a.bodies(), b.bodies())
        assert_interactions_equal(a.interactions(), b.interactions(), fields=("dn", "fn", "ft", "mom", "damp", "stick"))
        contacts += a.counts()["nactive"]
    assert contacts > 0 or n < 200  # the bodies met


@pytest.mark.parametrize("gap", [201.05, 201.25, 201.45])
@pytest.mark.parametrize("ndriven,heavy_min", [(1, None), (1, 1), (3, None), (3, 1)])
def test_limit_of_an_uncontrolled_driven_body(tmp_path, gap, ndriven, heavy_min):
    """A still driven sphere and a free one closing on it, whose allowances run
    out a fraction of a step apart: in the frame of the free bodies' mean
    velocity the driven sphere moves s = dt |mean| per step and the free one
    0.995 s, either's allowance is 100.5 s, and the pair is left off the list of
    step 2 at a gap a little above the two together, which is gone 101 steps
    later.  The driven sphere's bound passes its limit at just that step,
    which therefore has to test every entry again."""
    from rockable_amd.engine import Engine
    R, dt, u = 0.05, 1e-6, 0.1
    s = dt * u
    deck = D.Deck(dt=dt, tmax=1e3, interVerlet=1e3, interConf=1e3, DVerlet=5e-3, dVerlet=100.5 * s / 0.01,
                  density={0: 1000.0}, gravity=(0.0, 0.0, 0.0), nDriven=ndriven,
                  params=D.contact_params(1e5, 8e4, 0.25, 0.3))
    # the last driven sphere is the one that is met; the others are far away
    deck.bodies = [D.Body("S", pos=(0.0, 10.0 * (ndriven - 1 - k), 0.0)) for k in range(ndriven)]
    deck.bodies.append(D.Body("S", pos=(2 * R + (gap + 2 * 1.995) * s, 0.0, 0.0), vel=(-1.995 * u, 0.0, 0.0)))
    deck.bodies.append(D.Body("S", pos=(-2 * R - 5e-4, 0.0, 0.0), vel=(-0.005 * u, 0.0, 0.0)))
    path = D.write_deck(str(tmp_path), [D.sphere_shape("S", R)], deck)
    a, b = Engine(path), Engine(path)
    for e, skip in ((a, 1), (b, 0)):
        e.set_option("record_geometry", 0)
        e.set_option("skip_far", skip)
        if heavy_min is not None:
            e.set_option("heavy_min", heavy_min)
        e.update_nl()
        assert e.counts()["nlisted"] == 2
    for steps, active in ((102, 0), (1, 1), (5, 1)):
        a.step(steps)
        b.step(steps)
        assert b.counts()["nactive"] == active
        assert a.counts()["nactive"] == active
        assert_bodies_equal(a.bodies(), b.bodies())


@pytest.mark.parametrize("dims", [(8, 8, 4), (13, 13, 7), (32, 31, 24)])
def test_every_entry_listed(tmp_path, dims):
    """A squeezed lattice, every contact active: the parts of the list are full,
    with a lane for each of their entries and, past 65 536 entries, with fewer."""
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=dims, spacing_factor=1.9999, seed=7, vmax=0.01, nl="linkCells")
    path = D.write_deck(str(tmp_path), shapes, deck)
    a, b = Engine(path), Engine(path)
    for e, skip in ((a, 1), (b, 0)):
        e.set_option("record_geometry", 0)
        e.set_option("skip_far", skip)
        e.update_nl()
    for steps in (1, 30):
        a.step(steps)
        b.step(steps)
        c = a.counts()
        assert c["nactive"] == c["nlisted"] or steps > 1  # (half of them open as the lattice springs back)
        assert_bodies_equal(a.bodies(), b.bodies())
    assert (c["nlisted"] > 65536) == (dims[0] == 32)
    assert_interactions_equal(a.interactions(), b.interactions(), fields=("dn", "fn", "ft", "mom", "damp", "stick"))


def test_one_list_for_both_entry_buffers(tmp_path):
    """A rebuild that fills the other entry buffer for the first time takes no
    room for a second evaluation list: 640 bytes a listed entry (buffers are
    reserved for half as many again), 96 fewer than with one."""
    import ctypes
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=(60, 60, 30), spacing_factor=2.002, seed=3, vmax=0.0, nl="linkCells")
    e = Engine(D.write_deck(str(tmp_path), shapes, deck))
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    left = []
    for _ in range(2):
        e.update_nl()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        left.append(free.value)
    assert e.counts()["nlisted"] > 300000
    assert (left[0] - left[1]) / e.counts()["nlisted"] < 700
