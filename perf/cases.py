"""The calls whose speed a user of the engine feels, as timed cases.

Every case goes through the public entry points as a user's program does:
decks read by Engine.load_conf or load_batch, then step() and the read-out of
the state (bodies, and where a run monitors its contacts, the active
interactions and the statistics); and the training entry points of the
rebuild-interval network.  A pass advances the simulation by `steps` steps,
its neighbour-list rebuilds included, and reads the bodies once, as a run
that records every so many steps.

The bodies, laws and parameters are those of the repository's own
configurations (the 512 spheres on a lattice, the hull polyhedra of 8-14
points with the Avalanche law, the bonded clusters of 5 x 5 x 4 sphero-cubes,
the batches of sphere packings, the slope avalanche with the displacement
check), at sizes from a few hundred bodies to about 10^5, where a deck is
still read in about a second.
"""
import os
import shutil
import tempfile

import numpy as np

from rockable_amd import decks as D
from rockable_amd.engine import Engine, Mlp

G = 9.81
MLP_WEIGHTS = os.path.join("rockable_amd", "data", "rebuild_mlp.npy")
ROWS = ("pos", "Q", "vel", "vrot", "acc", "arot", "force", "moment")


def listed():
    return [
        # the repository's smallest configuration: 512 spheres dropping in a
        # box, Default law, every pair tested at a rebuild (launch latency)
        {"name": "spheres_512", "kind": "spheres", "bodies": 512, "nl": "bruteForce", "steps": 600},
        # a small polyhedral bed, an odd count, on the engine's default
        # options (every listed contact's geometry kept current), read out
        # with its active contacts and statistics as a monitored run does
        {"name": "bed_701_monitored", "kind": "bed", "bodies": 701, "law": "Default", "g": 100.0, "every": 100,
         "steps": 300, "monitor": True},
        {"name": "bed_6151_monitored", "kind": "bed", "bodies": 6151, "law": "Avalanche", "g": 100.0, "every": 100,
         "steps": 400, "monitor": True},
        # the settling stage of a pour: 400 g, a rebuild every 20 steps, so
        # that the neighbour list is a large part of it
        {"name": "settling_15007", "kind": "bed", "bodies": 15007, "law": "Avalanche", "g": 400.0, "every": 20,
         "steps": 200, "monitor": False},
        # the plain form of the headline configuration: 50 000 hulls,
        # Avalanche, linkCells, a rebuild every 100 steps
        {"name": "pour_50000", "kind": "bed", "bodies": 50000, "law": "Avalanche", "g": 100.0, "every": 100,
         "steps": 400, "monitor": False},
        # slope avalanches, rebuilt by the displacement check on the device:
        # fixed batches, and sized by the shipped network
        {"name": "slope_9973", "kind": "slope", "bodies": 9973, "network": False, "steps": 400},
        {"name": "slope_90001_network", "kind": "slope", "bodies": 90001, "network": True, "steps": 400},
        # bonded clusters that have hit a 35 degree plane (StickedLinks, the
        # host accounting each breakage)
        {"name": "bonds_12_clusters", "kind": "bonds", "clusters": 12, "steps": 300},
        {"name": "bonds_130_clusters", "kind": "bonds", "clusters": 130, "steps": 200},
        # independent sphere packings of uneven sizes in one engine
        {"name": "batch_24_packings", "kind": "batch", "packings": 24, "low": 500, "high": 5000, "steps": 400},
        # training of the rebuild network: loss and gradient over a whole set
        # of rebuild histories, and Adam over shuffled minibatches
        {"name": "network_gradient", "kind": "gradient", "samples": 20000},
        {"name": "network_training", "kind": "training", "samples": 4096, "batch": 256, "epochs": 3},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["spheres", "bed", "bed", "bed", "slope", "slope", "bonds", "batch", "gradient", "training"])
    if kind == "spheres":
        return {"kind": kind, "bodies": _log_int(rng, 200, 2000), "nl": rng.choice(["bruteForce", "linkCells"]),
                "steps": rng.randrange(300, 601)}
    if kind == "bed":
        monitor = rng.random() < 0.4
        g, every = rng.choice([(100.0, 100), (100.0, 100), (400.0, 20)])
        return {"kind": kind, "bodies": _log_int(rng, 500, 12000 if monitor else 50000),
                "law": rng.choice(["Default", "Avalanche"]), "g": g, "every": every,
                "steps": rng.randrange(150, 301), "monitor": monitor}
    if kind == "slope":
        return {"kind": kind, "bodies": _log_int(rng, 2000, 90000), "network": rng.random() < 0.5,
                "steps": rng.randrange(150, 401)}
    if kind == "bonds":
        return {"kind": kind, "clusters": _log_int(rng, 2, 130), "steps": rng.randrange(100, 201)}
    if kind == "batch":
        low = _log_int(rng, 300, 1000)
        return {"kind": kind, "packings": rng.randrange(4, 25), "low": low, "high": 5 * low,
                "steps": rng.randrange(150, 401)}
    if kind == "gradient":
        return {"kind": kind, "samples": _log_int(rng, 64, 20000)}
    return {"kind": kind, "samples": _log_int(rng, 600, 4096), "batch": rng.choice([128, 256]),
            "epochs": rng.randrange(1, 4)}


# --- decks -------------------------------------------------------------------
def _near_cube(n):
    nx = max(1, int(round(n ** (1.0 / 3.0))))
    return nx, nx, -(-n // (nx * nx))


def _spheres_deck(case, seed, where):
    """Spheres on a lattice with 1 % gaps falling into a box (the repository's
    first configuration a little closer, so that contacts form within a pass)."""
    shapes, deck = D.sphere_lattice_deck(dims=_near_cube(case["bodies"]), spacing_factor=2.02, seed=seed,
                                         nl=case["nl"], vmax=0.01)
    deck.bodies = deck.bodies[:deck.nDriven + case["bodies"]]
    return shapes, deck


def _settled_block(n, seed, law, where):
    """A block of n hulls settled by the engine in a small box: 2000 g, then
    400 g, then at rest under 100 g.  Returns the shapes, the deck it started
    from, the box width and the bodies."""
    width = float(np.ceil((n / 1.1) ** (1.0 / 3.0)))
    shapes, deck = D.compact_pour_deck(n_bodies=n, seed=seed, n_shapes=16, tilt_deg=3.0, gap_frac=0.0, vmax=0.5,
                                       law=law, interverlet_steps=20, width_in_sizes=width)
    eng = Engine(D.write_deck(where, shapes, deck, name="block.conf"))
    eng.set_option("record_geometry", 0)
    eng.update_nl()
    still = np.zeros((n + deck.nDriven, 3))
    for g, steps in ((2000.0, 9000), (400.0, 4000), (100.0, 3000)):
        eng.set_option("gravity_z", -g * G)
        eng.step(steps)
        if g <= 400.0:  # what still bounces is stopped
            eng.set_bodies(vel=still, vrot=still)
    b = {k: v[deck.nDriven:] for k, v in eng.bodies().items()}
    eng.close()
    return shapes, deck, 5e-3 * width, b


def _bed_deck(case, seed, where, law):
    """A bed of exactly `bodies` hulls: copies of a settled block side by side
    (the lowest bodies of the last copy fill the count), new walls around."""
    n = case["bodies"]
    block = min(n, 700)
    shapes, deck, width, b = _settled_block(block, seed, law, where)
    copies = -(-n // block)
    nx = int(np.ceil(np.sqrt(copies)))
    ny = -(-copies // nx)
    order = np.argsort(b["pos"][:, 2], kind="stable")  # a cut copy keeps its lowest bodies
    pick = np.concatenate([np.arange(block)] * (copies - 1) + [order[:n - block * (copies - 1)]])
    copy = np.minimum(np.arange(n) // block, copies - 1)
    pos = b["pos"][pick] + width * np.column_stack([copy % nx, copy // nx, np.zeros(n)])
    rng = np.random.default_rng(seed + 1)
    vel = rng.uniform(-0.01, 0.01, size=(n, 3))
    names = np.array([x.shape for x in deck.bodies[deck.nDriven:]])[pick]
    size = np.array([x.homothety for x in deck.bodies[deck.nDriven:]])[pick]
    hi = np.array([nx * width, ny * width, float(pos[:, 2].max()) + 5e-2])
    walls_shape, walls = D.box_walls(np.zeros(3), hi, 2.5e-4)
    deck.bodies = list(walls)
    deck.body_block = {"names": names, "group": np.zeros(n), "h": size, "pos": pos, "vel": vel, "Q": b["Q"][pick]}
    return walls_shape + shapes[1:], deck


def _bonds_deck(case, seed, where):
    """The bonded-cluster configuration for any number of clusters: the deck
    of one cluster repeated on a grid above the plane, the interface strengths
    drawn for each.  Written here as text, since a record per bond through
    the deck writer takes longer than the run."""
    m = case["clusters"]
    speed, clearance = 2.0, 1e-5
    shapes, deck = D.bonded_clusters_deck(n_clusters=1, seed=seed, speed=speed, clearance=clearance, plane_deg=35.0)
    rng = np.random.default_rng(seed)
    cubes = deck.bodies[1:]
    base = np.array([c.pos for c in cubes])
    per = len(cubes)
    side = int(np.ceil(np.sqrt(m)))
    pitch = (base.max(axis=0) - base.min(axis=0))[:2] + 5.5e-3 + 2e-3
    cell = np.arange(m)
    shift = np.zeros((m, 3))
    shift[:, 0] = (cell % side - 0.5 * side) * pitch[0]
    shift[:, 1] = (cell // side - 0.5 * side) * pitch[1]
    shift[:, 2] = -np.tan(np.radians(35.0)) * shift[:, 0]  # along the plane
    half = 1.5 * side * float(pitch.max()) + 0.1
    plane = D.square_plane_shape("PLANE", half, shapes[0].radius)
    bonds, links = deck.interactions, deck.interfaces
    deck.bodies, deck.interactions, deck.interfaces = deck.bodies[:1], [], []
    deck.body_block = {"names": "CUBE", "group": np.zeros(m * per), "cluster": np.repeat(cell, per),
                       "h": np.ones(m * per), "pos": (base[None] + shift[:, None]).reshape(-1, 3),
                       "vel": np.repeat(np.array([0.0, 0.0, -speed]) + rng.uniform(-0.1, 0.1, (m, 3)), per, axis=0),
                       "Q": np.tile([1.0, 0.0, 0.0, 0.0], (m * per, 1))}
    path = D.write_deck(where, [plane] + shapes[1:], deck)
    num = lambda xs: " ".join("%.16e" % x for x in xs)
    # one cluster's records as a format of the values that differ between clusters
    rec = "\n".join("%%d %%d %d %d %d %s %%.16e %%.16e %%.16e %s" % (t, a, b, num(r[5:9]), num(r[12:]))
                    for r in bonds for t, a, b in [r[2:5]])
    ij = np.array([r[:2] for r in bonds])
    at = np.array([r[9:12] for r in bonds])
    face = "\n".join("%%d %%d %d %.16e %s %%.16e %%.16e %s %s" % (
        len(f[4]), f[2], num(f[3][:3]), num(f[3][5:]), " ".join("%d %d %d" % q for q in f[4])) for f in links)
    pair = np.array([f[:2] for f in links])
    s2 = np.log(1.0 + 0.3 ** 2)
    out = ["Interactions %d" % (m * len(bonds))]
    for c in range(m):
        v = np.column_stack([ij + c * per, at + shift[c]]).astype(object)
        v[:, :2] = ij + c * per
        out.append(rec % tuple(v.ravel().tolist()))
    out.append("Interfaces %d" % (m * len(links)))
    for c in range(m):
        strength = np.exp(np.log(50.0) - 0.5 * s2 + np.sqrt(s2) * rng.standard_normal((len(links), 2)))
        v = np.empty((len(links), 4), dtype=object)
        v[:, :2] = pair + c * per
        v[:, 2:] = strength
        out.append(face % tuple(v.ravel().tolist()))
    with open(path) as fh:
        head = fh.read().rsplit("Interactions 0", 1)[0]
    with open(path, "w") as fh:
        fh.write(head + "\n".join(out) + "\n")
    return path


def _engine(case, seed):
    where = tempfile.mkdtemp(prefix="cases_")
    try:
        kind = case["kind"]
        if kind == "batch":
            # the packings' sizes and parameters belong to the case, their motion to the seed
            shapes, deck, info = D.batched_sphere_packings(case["packings"], (case["low"], case["high"]),
                                                           seed=case["packings"] + case["low"], spacing_factor=2.01,
                                                           dt=5e-7, en_range=(0.3, 0.9))
            vel = deck.body_block["vel"]
            vel[:] = np.random.default_rng(seed).uniform(-0.05, 0.05, size=vel.shape)
            paths = [D.write_deck(os.path.join(where, "p%d" % p), *D.single_packing_of(shapes, deck, info, p))
                     for p in range(case["packings"])]
            eng = Engine()
            eng.load_batch(paths)
        elif kind == "bonds":
            eng = Engine(_bonds_deck(case, seed, where))
        else:
            if kind == "spheres":
                shapes, deck = _spheres_deck(case, seed, where)
            elif kind == "bed":
                shapes, deck = _bed_deck(case, seed, where, case["law"])
                deck.gravity = (0.0, 0.0, -case["g"] * G)
                deck.interVerlet = case["every"] * deck.dt
            else:
                shapes, deck = _bed_deck(case, seed, where, "Avalanche")
                th = np.radians(30.0)
                deck.gravity = (G * np.sin(th), 0.0, -G * np.cos(th))
                deck.body_block["vel"][:, 0] += 1.0
                deck.interVerlet = 1e3
                deck.dynamic_update_nl = 1
                deck.disp_update_nl = 0.25 * deck.DVerlet
                deck.angle_update_nl = 180.0 / np.pi
            deck.tmax = 1e3
            eng = Engine(D.write_deck(where, shapes, deck))
    finally:
        shutil.rmtree(where, ignore_errors=True)
    if not case.get("monitor"):
        eng.set_option("record_geometry", 0)
    eng.update_nl()
    if case["kind"] == "bonds":
        eng.step(1500)  # through the impact, whose bursts of breakages differ from pass to pass
    return eng


# --- the network's data --------------------------------------------------------
def _samples(case, seed):
    """Guard features and targets as a rebuild history has them: features in
    [0, 1.2] growing over an interval, the logarithm of the steps left."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    life = np.exp(rng.uniform(np.log(5.0), np.log(400.0), size=n))
    used = rng.uniform(0.0, 1.0, size=n)
    x = rng.uniform(0.0, 1.0, size=(n, 16)) * (1.0 / life)[:, None] ** 0.5
    x[:, 0] = used
    x[:, 2] = 1.2 / life
    x[:, 9] = np.log1p((1.0 - used) * life) / 10.0
    x[:, 10] = np.log1p(used * life) / 10.0
    x[:, 11] = np.log1p(life) / 10.0
    x[:, 15] = 1.0
    t = np.log1p((1.0 - used) * life) + 0.05 * rng.standard_normal(n)
    return x.astype(np.float32), t.astype(np.float32)


def prepare(case, seed):
    if case["kind"] in ("gradient", "training"):
        net = Mlp(seed=1)
        net.set_params(np.load(MLP_WEIGHTS))
        x, t = _samples(case, seed)
        return {"case": case, "net": net, "x": x, "t": t}
    eng = _engine(case, seed)
    state = {"case": case, "engine": eng}
    if case.get("network"):
        net = Mlp(seed=1)
        net.set_params(np.load(MLP_WEIGHTS))
        eng.set_rebuild_model(net)
        state["net"] = net
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "gradient":
        loss, grad = state["net"].loss_grad(state["x"], state["t"])
        return {"loss": loss, "gradient": grad}
    if case["kind"] == "training":
        loss = state["net"].train(state["x"], state["t"], epochs=case["epochs"], batch=case["batch"], lr=2e-3)
        return {"loss": loss, "parameters": state["net"].params()}
    eng = state["engine"]
    eng.step(case["steps"])
    out = dict(eng.bodies())
    if case.get("monitor"):
        c = eng.interactions(active=True)
        room = 6 * case["bodies"]  # one table size for every pass, as a recorder has it
        for k in ("i", "j", "type", "isub", "jsub", "fn", "ft", "pos"):
            table = np.full((room,) + c[k].shape[1:], -1, dtype=c[k].dtype)
            table[:min(len(c), room)] = c[k][:room]
            out["contact_" + k] = table
        s = eng.stats()
        out["coordination"], out["kinetic"] = s["coordination"], s["kinetic_translational"]
    return out


# --- the work of a pass ----------------------------------------------------------
def work(case):
    """Bytes that a pass cannot do without.  Per step: each body's pose,
    velocities, accelerations and resultants read and written once (26
    doubles read, 25 written: 408 bytes) and its inertia and mass (32), and
    each active contact's state (fn, ft, mom, dn) read and written (128).
    Per rebuild: each body's pose and each listed contact's key and state
    (body pair, sub-elements, history) read and written once.  The counts per
    body are those that these packings have."""
    kind = case["kind"]
    per = 16 * 64 + 64 + 64 * 64 + 64 + 64 + 1
    if kind == "gradient":
        n = case["samples"]
        return {"bytes": 4 * (17 * n + 2 * per + 1), "flops": 6 * n * (16 * 64 + 64 * 64 + 64)}
    if kind == "training":
        n = case["samples"] // case["batch"] * case["batch"] * case["epochs"]
        return {"bytes": 4 * (17 * n + 4 * per), "flops": 6 * n * (16 * 64 + 64 * 64 + 64)}
    if kind == "batch":
        bodies = case["packings"] * (case["high"] - case["low"]) / np.log(case["high"] / case["low"])
    else:
        bodies = case["clusters"] * 100 if kind == "bonds" else case["bodies"]
    active, known = {"spheres": (0.2, 3.0), "batch": (0.1, 3.0), "bed": (1.6, 20.0), "slope": (0.5, 20.0),
                     "bonds": (9.0, 32.0)}[kind]
    every = case.get("every", 50 if kind == "slope" else 100)
    per_step = bodies * (440 + 128 * active)
    per_rebuild = bodies * (2 * 96 * known + 128)
    flops = bodies * (300 + 400 * active)
    return {"bytes": case["steps"] * (per_step + per_rebuild / every) + 200 * bodies, "flops": case["steps"] * flops}


# --- the same in numpy -------------------------------------------------------------
def _network_gradient(params, x, t):
    """Loss and gradient of the 16-64-64-1 tanh network, in 64 bits."""
    p = params.astype(np.float64)
    w1, b1, w2, b2, w3, b3 = np.split(p, np.cumsum([1024, 64, 4096, 64, 64]))
    w1, w2 = w1.reshape(64, 16), w2.reshape(64, 64)
    x, t = x.astype(np.float64), t.astype(np.float64)
    h1 = np.tanh(x @ w1.T + b1)
    h2 = np.tanh(h1 @ w2.T + b2)
    r = h2 @ w3 + b3[0] - t
    e = 2.0 * r / len(t)
    d2 = e[:, None] * w3 * (1.0 - h2 * h2)
    d1 = (d2 @ w2) * (1.0 - h1 * h1)
    grad = [(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), e @ h2, [e.sum()]]
    return float(np.mean(r * r)), np.concatenate(grad)


def _spheres_by_numpy(case, seed):
    """The sphere case in numpy: velocity Verlet, Default law between spheres
    and with the five walls.  The spheres stay inside the box, so a wall is
    its inner plane; rotations matter through the friction alone, but the
    quaternions are integrated too."""
    shapes, deck = _spheres_deck(case, seed, None)
    nd, R = deck.nDriven, shapes[-1].radius
    bodies = deck.bodies[nd:]
    n, dt = len(bodies), deck.dt
    par = {p[0]: p[3] for p in deck.params}
    kn, kt, mu, en2 = par["knContact"], par["ktContact"], par["muContact"], par["en2Contact"]
    m = 2700.0 * shapes[-1].volume
    inertia = m * shapes[-1].inertia_mass[0]
    rate = -0.5 * np.log(en2) / np.sqrt((0.5 * np.log(en2)) ** 2 + np.pi ** 2)
    g = np.array(deck.gravity)
    x = np.array([b.pos for b in bodies])
    v = np.array([b.vel for b in bodies])
    q = np.tile([1.0, 0.0, 0.0, 0.0], (n, 1))
    w, acc, arot = np.zeros((n, 3)), np.tile(g, (n, 1)), np.zeros((n, 3))
    # walls: a point of the inner plane, the inward normal, the centre
    wr = shapes[0].radius
    normal = np.array([[0, 0, 1.0], [1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0]])
    centre = np.array([b.pos for b in deck.bodies[:nd]])
    ft_w = np.zeros((nd, n, 3))
    pi, pj = np.triu_indices(n, 1)
    ai = aj = np.zeros(0, dtype=int)
    ft_p = np.zeros((0, 3))

    def hamilton(a, b):  # (0, a) times the quaternions b
        return np.column_stack([-(a * b[:, 1:]).sum(1), a * b[:, :1] + np.cross(a, b[:, 1:])])

    def friction(old, vn, vel, nrm, kn_dn):
        vt = vel - vn[:, None] * nrm
        f = old + kt * dt * vt
        cap = mu * kn_dn
        s = np.sqrt((f * f).sum(1))
        over = (s > 0) & (s >= cap)
        return np.where(over[:, None], f * (cap / np.where(s > 0, s, 1.0))[:, None], f)

    for k in range(case["steps"]):
        if k % 100 == 0:  # the neighbour list: a contact's friction lasts while its pair stays listed
            old = {(a, b): f for a, b, f in zip(ai, aj, ft_p)}
            near = np.nonzero(((x[pi] - x[pj]) ** 2).sum(1) <= (2 * R + deck.dVerlet) ** 2)[0]
            ai, aj = pi[near], pj[near]
            ft_p = np.array([old.get((a, b), np.zeros(3)) for a, b in zip(ai, aj)]).reshape(-1, 3)
            for b in range(nd):
                ft_w[b, (x - centre[b]) @ normal[b] - (R + wr) > deck.dVerlet] = 0.0
        x = x + (dt * v + 0.5 * dt * dt * acc)
        v = v + 0.5 * dt * acc
        dq = 0.5 * hamilton(w, q)
        ddq = 0.5 * hamilton(arot, q) + 0.5 * hamilton(w, dq)
        q = q + dt * dq + 0.5 * dt * dt * ddq
        q /= np.sqrt((q * q).sum(1))[:, None]
        w = w + 0.5 * dt * arot
        F, M = np.zeros((n, 3)), np.zeros((n, 3))
        wall_f, wall_m = np.zeros((nd, 3)), np.zeros((nd, 3))
        r = x[ai] - x[aj]
        dist = np.sqrt((r * r).sum(1))
        dn = dist - 2 * R
        hit = dn < 0
        nrm = r / dist[:, None]
        c = x[ai] - (R + 0.5 * dn)[:, None] * nrm
        vel = (v[aj] - np.cross(c - x[aj], w[aj])) - (v[ai] - np.cross(c - x[ai], w[ai]))
        vn = (vel * nrm).sum(1)
        fn = np.maximum(-kn * dn + rate * 2.0 * np.sqrt(kn * 0.5 * m) * vn, 0.0)
        ft_p = np.where(hit[:, None], friction(ft_p, vn, vel, nrm, np.abs(kn * dn)), ft_p)
        f = np.where(hit[:, None], fn[:, None] * nrm + ft_p, 0.0)
        np.add.at(F, ai, f)
        np.add.at(F, aj, -f)
        np.add.at(M, ai, np.cross(c - x[ai], f))
        np.add.at(M, aj, np.cross(c - x[aj], -f))
        for b in range(nd):  # the sphere is the second body of the pair in the engine's order
            dist = (x - centre[b]) @ normal[b]
            dn = dist - (R + wr)
            hit = dn < 0
            if not hit.any():
                continue
            nw = np.tile(normal[b], (n, 1))
            c = x - (R + 0.5 * dn)[:, None] * nw
            vel = -(v - np.cross(c - x, w))
            vn = (vel * nw).sum(1)
            fn = np.maximum(-kn * dn + rate * 2.0 * np.sqrt(kn * m) * vn, 0.0)
            ft_w[b] = np.where(hit[:, None], friction(ft_w[b], vn, vel, nw, np.abs(kn * dn)), ft_w[b])
            f = np.where(hit[:, None], fn[:, None] * nw + ft_w[b], 0.0)
            F += f
            M += np.cross(c - x, f)
            wall_f[b] = -f.sum(0)
            wall_m[b] = np.cross(c - centre[b], -f).sum(0)
        acc = F / m + g
        arot = M / inertia
        v = v + 0.5 * dt * acc
        w = w + 0.5 * dt * arot
    still = np.zeros((nd, 3))
    wall_q = np.array([b.Q for b in deck.bodies[:nd]])
    return {"pos": np.vstack([centre, x]), "Q": np.vstack([wall_q, q]), "vel": np.vstack([still, v]),
            "vrot": np.vstack([still, w]), "acc": np.vstack([still, acc]), "arot": np.vstack([still, arot]),
            "force": np.vstack([wall_f, F]), "moment": np.vstack([wall_m, M])}


def exact(case, seed):
    """The network's gradient and a run of spheres in numpy, in 64 bits.  The
    engine's other runs are hundreds of steps of polyhedra: a numpy step of
    those takes longer than the bound allows, and they are 64-bit
    computations already."""
    if case["kind"] == "gradient":
        loss, grad = _network_gradient(np.load(MLP_WEIGHTS), *_samples(case, seed))
        return {"loss": loss, "gradient": grad}
    if case["kind"] == "spheres" and case["bodies"] <= 600:
        return _spheres_by_numpy(case, seed)
    return None
