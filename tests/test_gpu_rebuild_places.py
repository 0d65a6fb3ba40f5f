"""Places by counts in the neighbour-list rebuild: a body's directed groups
and its entries as second body are placed by loops over short segments and by
bitmaps over long ones, in windows of 2^18 values."""
import numpy as np
import pytest

from tests.test_gpu_parity import assert_bodies_equal, assert_interactions_equal

pytestmark = pytest.mark.gpu


def _engine(tmp_path, dims, spacing=2.002, **kw):
    from rockable_amd import decks as D
    from rockable_amd.engine import Engine
    shapes, deck = D.sphere_lattice_deck(dims=dims, spacing_factor=spacing, seed=5, nl="linkCells", **kw)
    path = D.write_deck(str(tmp_path), shapes, deck)
    return Engine(path), path


@pytest.mark.parametrize("dims", [(1, 1, 1), (16, 16, 1), (16, 32, 1), (27, 19, 1), (40, 40, 2)])
def test_lists_match_oracle(tmp_path, dims):
    """Floors of 1, 256, 512, 513 and 1 600 spheres, so segments of both kinds
    and at the line between them, rebuilt from an empty list and from their
    own: the lists and the motion equal the serial oracle's bit for bit."""
    from oracle.rk_oracle import Oracle
    e, path = _engine(tmp_path, dims)
    o = Oracle(path)
    for _ in range(3):
        e.update_nl()
        o.update_nl()
        assert_interactions_equal(e.interactions(), o.interactions(), fields=("dn", "fn", "ft", "mom", "damp", "stick"))
        e.step(5)
        o.run_steps(5)
        assert_bodies_equal(e.bodies(), o.bodies())


def test_windows_past_the_first(tmp_path):
    """265 200 spheres on a floor: body indices and entry indices beyond one
    window.  The list is that of the lattice: every sphere with its axis
    neighbours, with the floor and with the walls, in ascending order, each
    pair once and unchanged by a rebuild; the resultants of the contacts that
    form, on bodies and in slots past the first window, equal the serial sums
    of the heavy-body kernel."""
    dims = (340, 260, 3)
    e, _ = _engine(tmp_path, dims, vmax=0.05)
    e.set_option("exact_sums", 1)
    e.update_nl()
    a = e.interactions()
    e.update_nl()
    assert_interactions_equal(e.interactions(), a)
    nw, (nx, ny, nz) = 5, dims
    i, j = a["i"].astype(np.int64), a["j"].astype(np.int64)
    key = i * (nw + nx * ny * nz) + j
    assert np.all(np.diff(key) >= 0)
    ss = (i >= nw) & (j >= nw)
    idx = np.arange(nx * ny * nz).reshape(nx, ny, nz) + nw
    want = np.concatenate([np.stack([p.ravel(), q.ravel()], 1) for p, q in
                           ((idx[1:], idx[:-1]), (idx[:, 1:], idx[:, :-1]), (idx[:, :, 1:], idx[:, :, :-1]))])
    want = np.unique(np.sort(want, axis=1), axis=0)
    got = np.sort(np.stack([i[ss], j[ss]], 1), axis=1)
    assert len(got) == len(want)
    assert np.array_equal(np.unique(got, axis=0), want)
    floor = np.unique(np.concatenate([i[(j < nw)], j[(i < nw)]]))
    edge = np.unique(np.concatenate([idx[:, :, 0].ravel(), idx[0].ravel(), idx[-1].ravel(), idx[:, 0].ravel(),
                                     idx[:, -1].ravel()]))
    assert np.array_equal(floor, edge)
    b, _ = _engine(tmp_path, dims, vmax=0.05)
    b.set_option("exact_sums", 1)
    b.set_option("heavy_min", 1)
    b.update_nl()
    b.update_nl()
    for x in (e, b):
        x.step(60)
    act = e.interactions()
    act = np.nonzero((act["dn"] < 0) & (act["i"] > 2 ** 18))[0]
    assert len(act) > 100 and act.max() > 2 ** 18
    assert_bodies_equal(e.bodies(), b.bodies())


def test_more_pairs_left_than_the_last_rebuild(tmp_path):
    """The narrow phase's grid comes from the last rebuild's count of the pairs
    left to it: hulls far apart first, so that the second rebuild has thousands
    more than the grid covers, against an engine that starts from the second
    state."""
    from rockable_amd import decks as D
    from rockable_amd.engine import Engine
    shapes, deck = D.compact_pour_deck(n_bodies=2000, seed=2, n_shapes=8, box_in_sizes=(12, 12, 60))
    deck.DVerlet = deck.dVerlet = 3e-3  # every pair of neighbours listed
    path = D.write_deck(str(tmp_path), shapes, deck)
    a, b = Engine(path), Engine(path)
    near = a.bodies()["pos"].copy()
    far = near * 4.0
    a.set_bodies(pos=far)
    a.update_nl()
    few = a.counts()["nlisted"]
    a.set_bodies(pos=near)
    a.update_nl()
    b.set_bodies(pos=near)
    b.update_nl()
    assert b.counts()["nlisted"] > few + 2000
    keys = ("i", "j", "type", "isub", "jsub")
    x, y = a.interactions(), b.interactions()
    have = set(zip(*(x[k].tolist() for k in keys)))
    want = set(zip(*(y[k].tolist() for k in keys)))
    assert want <= have
    kept = have - want  # entries of the far list that no near test looks at again stay listed
    assert len(kept) <= few
