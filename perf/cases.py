"""The performance cases: what programs have the engine do, through its public entry points.

Every case is a plain dict.  Its `kind` says what one pass is:

  run       Engine.run in chunks of `every` steps with the species counted after each chunk (a recorder's
            stride), then the particles read back
  actions   the same steps as separate actions (integrate, neighbour list, reactions, neighbour list,
            forces) with the energy read after each, as a kernel plug-in is driven, then the particles
  forces    one force evaluation, the energy and the forces read back
  rdf       one radial distribution of all particles
  ensemble  uneven replicas stepped together in one engine, their counts and particles read back
  serve     requests of uneven size and length admitted to a shared engine, stepped in intervals, read
            back and retired as they finish

The chemistries are those of the benchmark configurations: `ab` (harmonic repulsion, A+B<->C), `ab_weak`
(with the A-A weak interaction, whose cutoff is twice the others') and `chains` (bead chains with bonds,
angles and dihedrals among Lennard-Jones crowders, enzymatic binding).  `headroom` is the particle budget
a program asks for at add_replica, as a multiple of what it uploads.

`exact` restates the same steps in NumPy, in 64 bits: the noise and the draws are the engine's documented
Philox counters, so the trajectories are comparable particle by particle.
"""
import functools
import math

import numpy as np

from readdy_amd import Engine, workloads
from readdy_amd import _lib as L

HANDLERS = {"ua": L.HANDLER_UA, "gillespie": L.HANDLER_GILLESPIE}
DIFFUSION = {"ab": [1.0, 1.0, 0.5], "ab_weak": [1.0, 1.0, 0.5], "chains": [0.5, 1.0, 1.0]}
BEADS = 50  # beads of a chain


def chemistry(chem):
    """(pair potentials, reactions) of a chemistry."""
    if chem == "chains":
        return workloads.potentials(L), workloads.reactions(L, 0.01)
    pots, rxs = workloads.c1_chemistry(L)
    return (pots if chem == "ab_weak" else [p for p in pots if p[0] == L.POT_HARMONIC_REPULSION]), rxs


def listed():
    return [
        # a program that looks at every step of a small system: latency and launches are all of it
        dict(name="step_500", kind="run", chem="ab", n=500, density=0.25, handler="ua", dt=0.01, steps=1, every=1,
             headroom=2),
        # the plain small system with its species counts recorded every ten steps
        dict(name="run_2k", kind="run", chem="ab", n=2000, density=0.25, handler="ua", dt=0.01, steps=100, every=10,
             headroom=4),
        # a served request's system on an engine of its own, with the other handler
        dict(name="run_30k_gillespie", kind="run", chem="ab_weak", n=30011, density=0.125, handler="gillespie",
             dt=0.005, steps=100, every=50, headroom=2),
        # a crowded mid-size system
        dict(name="run_200k_dense", kind="run", chem="ab", n=200000, density=0.6, handler="ua", dt=0.01, steps=200,
             every=100, headroom=1),
        # the headline system
        dict(name="run_1m", kind="run", chem="ab_weak", n=1000000, density=0.125, handler="ua", dt=0.005, steps=500,
             every=250, headroom=1),
        # bead chains with bonded terms among crowders, small and large
        dict(name="chains_4k", kind="run", chem="chains", n=4000, density=0.244, handler="gillespie", dt=2e-4,
             steps=20, every=10, headroom=2),
        dict(name="chains_200k", kind="run", chem="chains", n=200000, density=0.244, handler="gillespie", dt=2e-4,
             steps=50, every=50, headroom=2),
        # a plug-in's loop: every action its own call, the energy observed each step
        dict(name="actions_20k", kind="actions", chem="ab_weak", n=20003, density=0.25, handler="ua", dt=0.005,
             steps=10, headroom=2),
        # one force evaluation of a large state (a forces / energy observable, a minimiser)
        dict(name="forces_300k", kind="forces", chem="ab_weak", n=300000, density=0.125, headroom=1),
        # the pair-correlation observable of the headline system
        dict(name="rdf_1m", kind="rdf", chem="ab_weak", n=1000000, density=0.125, bins=100, r_max=5.0, headroom=1),
        # a batched ensemble of uneven replicas
        dict(name="ensemble_64", kind="ensemble", chem="ab", replicas=64, n_min=500, n_max=50000, density=0.25,
             handler="ua", dt=0.01, steps=200, cell=2.0),
        # continuous batching of a dozen requests
        dict(name="serve_12", kind="serve", chem="ab_weak", replicas=12, n_min=1000, n_max=50000, density=0.125,
             dt=0.005, steps_min=40, steps_max=160, interval=40),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "chains", "actions", "forces", "rdf", "ensemble", "serve"])
    chem = rng.choice(["ab", "ab_weak"])
    density = round(rng.uniform(0.1, 0.7), 3)
    headroom = rng.choice([1, 2, 4])
    handler = rng.choice(["ua", "gillespie"])
    dt = rng.choice([0.005, 0.01])
    if kind == "run":
        n = _log_uniform(rng, 500, 1000000)
        steps = max(1, min(_log_uniform(rng, 1, 500), int(6e7 / (n * density))))
        return dict(kind="run", chem=chem, n=n, density=density, handler=handler, dt=dt, steps=steps,
                    every=rng.randint(1 + steps // 8, steps), headroom=headroom)
    if kind == "chains":
        steps = _log_uniform(rng, 1, 50)
        return dict(kind="run", chem="chains", n=2 * BEADS * _log_uniform(rng, 8, 2000), density=0.244,
                    handler=handler, dt=2e-4, steps=steps, every=rng.randint(1 + steps // 8, steps),
                    headroom=headroom)
    if kind == "actions":
        return dict(kind="actions", chem=chem, n=_log_uniform(rng, 500, 200000), density=density, handler=handler,
                    dt=dt, steps=rng.randint(1, 20), headroom=headroom)
    if kind == "forces":
        if rng.random() < 0.3:
            return dict(kind="forces", chem="chains", n=2 * BEADS * _log_uniform(rng, 8, 2000), density=0.244,
                        headroom=headroom)
        return dict(kind="forces", chem=chem, n=_log_uniform(rng, 500, 1000000), density=density, headroom=headroom)
    if kind == "rdf":
        r_max = round(rng.uniform(1.0, 5.0), 2)
        n = _log_uniform(rng, 500, 1000000)
        return dict(kind="rdf", chem=chem, n=max(500, min(n, int(3e7 / (density * r_max ** 3)))), density=density,
                    bins=_log_uniform(rng, 10, 1000), r_max=r_max, headroom=headroom)
    if kind == "ensemble":
        return dict(kind="ensemble", chem="ab", replicas=_log_uniform(rng, 2, 64), n_min=500,
                    n_max=_log_uniform(rng, 2000, 50000), density=round(rng.uniform(0.1, 0.4), 3), handler=handler,
                    dt=dt, steps=_log_uniform(rng, 10, 200), cell=rng.choice([1.0, 2.0]))
    return dict(kind="serve", chem="ab_weak", replicas=rng.randint(2, 12), n_min=1000,
                n_max=_log_uniform(rng, 5000, 50000), density=0.125, dt=0.005, steps_min=20,
                steps_max=rng.randint(40, 160), interval=rng.randint(20, 60))


# ---- inputs -------------------------------------------------------------------------------------------
def _box(n, density):
    return (n / density) ** (1.0 / 3.0)


@functools.lru_cache(maxsize=2)
def _chain_geometry(n, box):
    """One chain system of n particles, half of them beads (built once per size: it takes seconds)."""
    return workloads.system(n // 2 // BEADS, BEADS, n - n // 2, box, 2)


def _system(case, seed):
    """(positions, types, bonded index lists or None, box) of a case's system."""
    box = _box(case["n"], case["density"])
    rng = np.random.default_rng([seed, case["n"]])
    if case["chem"] == "chains":
        pos, types, bonds, angles, dihedrals = _chain_geometry(case["n"], box)
        # another placement of the same geometry: axes in another order, shifted through the boundary
        pos = (pos[:, rng.permutation(3)] + rng.random(3) * box + box / 2) % box - box / 2
        return pos, types, (bonds, angles, dihedrals), box
    pos = (rng.random((case["n"], 3)) - 0.5) * box
    types = rng.choice(np.array([0, 1, 2], dtype=np.uint32), case["n"], p=[0.4, 0.4, 0.2])
    return pos, types, None, box


def _replicas(case, seed):
    """(n, box, seed, handler, steps) of the replicas of an ensemble or the requests of a trace: sizes (and a
    request's length and handler) log-uniform and of the case, the states of the seed."""
    rng = np.random.default_rng(case["replicas"])
    r = case["replicas"]
    n = np.exp(rng.uniform(math.log(case["n_min"]), math.log(case["n_max"]), r)).astype(int)
    n[0], n[-1] = case["n_max"], case["n_min"]
    if case["kind"] == "serve":
        handler = np.where(rng.random(r) < 0.5, "ua", "gillespie")
        steps = np.exp(rng.uniform(math.log(case["steps_min"]), math.log(case["steps_max"]), r)).astype(int)
    else:
        handler, steps = [case["handler"]] * r, [case["steps"]] * r
    return [(int(n[k]), _box(int(n[k]), case["density"]), seed * 4096 + k, str(handler[k]), int(steps[k]))
            for k in range(r)]


def _replica_state(n, box, seed):
    rng = np.random.default_rng(seed)
    return (rng.random((n, 3)) - 0.5) * box, rng.choice(np.array([0, 1, 2], dtype=np.uint32), n, p=[0.4, 0.4, 0.2])


def _fill(e, box, seed, pos, types, terms, headroom):
    r = e.add_replica([box] * 3, (1, 1, 1), seed=seed, max_particles=int(headroom * len(types)))
    e.set_particles(r, pos, types)
    if terms:
        e.set_bonds(r, terms[0], 100.0, 1.0)
        e.set_angles(r, terms[1], 10.0, np.pi)
        e.set_dihedrals(r, terms[2], 1.0, 3, 0.0)
    return r


def prepare(case, seed):
    pots, rxs = chemistry(case["chem"])
    kw = dict(potentials=pots, reactions=rxs)
    s = {"case": case}
    if case["kind"] in ("ensemble", "serve"):
        reps = _replicas(case, seed)
        total = sum(r[0] for r in reps)
        cell = case.get("cell", 2.0)
        cells = sum(max(1, int(r[1] // cell)) ** 3 for r in reps)
        lam = total / cells
        cap = max(8, int(math.ceil(lam + 7.0 * math.sqrt(lam) + 6.0)) // 4 * 4 + 4)
        # a server's pools are larger than what it holds at one time
        room = 1 if case["kind"] == "ensemble" else 2
        e = Engine(3, DIFFUSION[case["chem"]], nl_cutoff=cell, bin_capacity=cap, max_replicas=len(reps),
                   max_cells=room * cells, max_particles=2 * room * total + 4096, **kw)
        data = [_replica_state(n, box, sd) for n, box, sd, _, _ in reps]
        s.update(engine=e, reps=reps, data=data)
        if case["kind"] == "ensemble":
            s["ids"] = [_fill(e, box, sd, p, t, None, 2) for (n, box, sd, _, _), (p, t) in zip(reps, data)]
        return s
    pos, types, terms, box = _system(case, seed)
    e = Engine(3, DIFFUSION[case["chem"]], topology_flavor=[1, 0, 0] if terms else None, **kw)
    s.update(engine=e, r=_fill(e, box, seed, pos, types, terms, case["headroom"]))
    if case["kind"] == "actions":
        e.calculate_forces()  # the loop's initial forces
    return s


# ---- one pass -----------------------------------------------------------------------------------------
def _rows(n):
    """A+C and B+C are conserved: 0.4 / 0.4 / 0.2 of n can at most become 1.2 n particles (and the draw's spread)."""
    return int(1.2 * n + 6 * math.sqrt(n)) + 16


def _frame(parts, rows):
    """The particles of all parts in a frame of `rows` rows, as a program keeps one for a varying count."""
    out = {"positions": np.zeros((rows, 3)), "types": np.full(rows, -1, dtype=np.int64),
           "handles": np.full(rows, -1, dtype=np.int64)}
    at = 0
    for part in parts:
        for a, v in zip(out.values(), part):
            a[at:at + len(v)] = v
        at += len(part[1])
    return out


def _run_run(s, c):
    e, r, h = s["engine"], s["r"], HANDLERS[c["handler"]]
    counts, done = [], 0
    while done < c["steps"]:
        k = min(c["every"], c["steps"] - done)
        e.run(h, c["dt"], k, graph=True)
        counts.append(e.count_types(r + 1)[r])
        done += k
    return dict(_frame([e.get_particles(r)], _rows(c["n"])), counts=np.array(counts, dtype=np.int64))


def _run_actions(s, c):
    e, r, h = s["engine"], s["r"], HANDLERS[c["handler"]]
    energies = []
    for _ in range(c["steps"]):
        e.integrate(c["dt"])
        e.update_neighbor_list()
        e.react(h, c["dt"])
        e.update_neighbor_list()
        e.calculate_forces()
        energies.append(e.energy(r))
    return dict(_frame([e.get_particles(r)], _rows(c["n"])), energies=np.array(energies))


def _run_forces(s, c):
    e, r = s["engine"], s["r"]
    e.calculate_forces()
    energy = e.energy(r)
    forces, handles = e.get_forces(r)
    return {"forces": forces, "handles": handles.astype(np.int64), "energy": energy}


def _run_rdf(s, c):
    counts, n_from = s["engine"].rdf_counts(s["r"], np.linspace(0.0, c["r_max"], c["bins"] + 1), [0, 1, 2], [0, 1, 2])
    return {"counts": counts.astype(np.int64), "n_from": int(n_from)}


def _run_ensemble(s, c):
    e, ids = s["engine"], s["ids"]
    e.run(HANDLERS[c["handler"]], c["dt"], c["steps"], graph=True)
    counts = e.count_types(max(ids) + 1)[ids]
    rows = sum(_rows(rep[0]) for rep in s["reps"])
    return dict(_frame([e.get_particles(r) for r in ids], rows), counts=counts.astype(np.int64))


def _run_serve(s, c):
    e = s["engine"]
    active, final = {}, {}
    for k, ((n, box, seed, handler, steps), (pos, types)) in enumerate(zip(s["reps"], s["data"])):
        r = _fill(e, box, seed, pos, types, None, 2)
        e.set_handler(r, HANDLERS[handler])
        e.set_steps(r, steps)
        active[r] = [k, steps]
    observed = []
    while active:
        k = min(c["interval"], max(left for _, left in active.values()))
        e.run(L.HANDLER_UA, c["dt"], k, graph=True)
        counts = e.count_types(max(active) + 1)
        for r in list(active):
            observed.append(counts[r])
            active[r][1] -= min(k, active[r][1])
            if active[r][1] == 0:
                final[active[r][0]] = e.get_particles(r)
                e.remove_replica(r)
                del active[r]
    rows = sum(_rows(rep[0]) for rep in s["reps"])
    return dict(_frame([final[k] for k in sorted(final)], rows), counts=np.array(observed, dtype=np.int64))


_RUN = {"run": _run_run, "actions": _run_actions, "forces": _run_forces, "rdf": _run_rdf, "ensemble": _run_ensemble,
        "serve": _run_serve}


def run(state):
    return _RUN[state["case"]["kind"]](state, state["case"])


# ---- work, tolerance ----------------------------------------------------------------------------------
STATE = 32.0         # bytes of a particle's state: FP64 position, species, id
PAIR = 40.0          # operations of a pair: displacement, minimum image, square, force, two sums
TERMS = 17.2 * 2     # bytes of a chain bead's static index lists and parameters


def _pairs_per_particle(case):
    """Neighbours of a particle inside its potentials' cutoffs (a uniform state)."""
    if case["chem"] == "chains":
        return 4.2 * 2.5 ** 3 * case["density"] * 0.75
    return 4.2 * case["density"] * (1.0 + (0.16 * 7.0 if case["chem"] == "ab_weak" else 0.0))


def work(case):
    kind = case["kind"]
    if kind in ("ensemble", "serve"):
        reps = _replicas(case, 0)
        n = sum(r[0] for r in reps)
        steps = sum(r[0] * r[4] for r in reps) / n
    else:
        n, steps = case["n"], case.get("steps", 1)
    if kind == "rdf":
        pairs = n * 4.2 * case["density"] * case["r_max"] ** 3
        return {"bytes": n * STATE + 8.0 * case["bins"], "flops": 12.0 * pairs}
    flops = n * steps * (_pairs_per_particle(case) * PAIR + 100.0)
    if kind == "forces":
        return {"bytes": n * (STATE + 28.0), "flops": flops}
    per = 2 * STATE + (TERMS / 2 if case["chem"] == "chains" else 0.0)
    return {"bytes": n * (steps * per + STATE), "flops": flops}


def tolerance(case):
    if case["kind"] == "rdf":
        return "exact"
    if case["kind"] == "forces":
        return {"rel": 5e-7}  # FP32 pair arithmetic, summed exactly: 1.1e-7 measured
    if case["chem"] == "chains":
        # straight angles make the dihedrals of the chains ill-conditioned: a rounding grows to 1e-2 on a few
        # beads within fifty steps
        return {"rel": 1e-3, "differ": 1e-3}
    # FP32 pair forces and noise moving FP64 positions: up to 9e-8 in a hundred steps, 2.1e-7 in an energy
    return {"rel": 1e-6 if case["kind"] == "actions" else 4e-7, "differ": 1e-4}


# ---- the same in NumPy, 64 bits -------------------------------------------------------------------------
def _philox(c0, c1, c2, c3, seed):
    """Philox4x32-10 (Salmon et al., SC'11), counters as arrays."""
    c = [np.broadcast_to(np.asarray(x, dtype=np.uint64), np.broadcast(c0, c1, c2, c3).shape) for x in (c0, c1, c2, c3)]
    k0, k1 = int(seed) & 0xFFFFFFFF, (int(seed) >> 32) & 0xFFFFFFFF
    low, half = np.uint64(0xFFFFFFFF), np.uint64(32)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> half) ^ c[1] ^ np.uint64(k0), p1 & low, (p0 >> half) ^ c[3] ^ np.uint64(k1), p0 & low]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c


def _u53(a, b):
    return ((a >> np.uint64(5)).astype(float) * 67108864.0 + (b >> np.uint64(6)).astype(float)) / 2.0 ** 53


def _box_muller(v):
    r0, r1 = np.sqrt(-2.0 * np.log(v[0])), np.sqrt(-2.0 * np.log(v[2]))
    return np.stack([r0 * np.cos(2 * np.pi * v[1]), r0 * np.sin(2 * np.pi * v[1]), r1 * np.cos(2 * np.pi * v[3])], -1)


def _image(d, box):
    return d - box * (d > 0.5 * box) + box * (d <= -0.5 * box)


def _wrap(x, box):
    while np.any(hi := x >= 0.5 * box):
        x = x - box * hi
    while np.any(lo := x < -0.5 * box):
        x = x + box * lo
    return x


def _pairs(pos, box, cut):
    """Yields (i, j, x_j - x_i, squared distance) of the unordered pairs closer than cut."""
    n, dims = len(pos), int(box // cut)
    if dims < 3:
        i, j = np.triu_indices(n, 1)
        blocks = [(i, j)]
    else:
        c = np.minimum((np.floor((pos + 0.5 * box) / (box / dims))).astype(np.int64), dims - 1)
        key = (c[:, 0] * dims + c[:, 1]) * dims + c[:, 2]
        order = np.argsort(key, kind="stable")
        start = np.searchsorted(key[order], np.arange(dims ** 3 + 1))

        def expand():
            for a in (-1, 0, 1):
                for b in (-1, 0, 1):
                    for z in (-1, 0, 1):
                        if (a, b, z) < (0, 0, 0):
                            continue
                        for lo in range(0, n, 1 << 17):
                            me = order[lo:lo + (1 << 17)]
                            k = (((c[me, 0] + a) % dims) * dims + (c[me, 1] + b) % dims) * dims + (c[me, 2] + z) % dims
                            cnt = start[k + 1] - start[k]
                            i = np.repeat(me, cnt)
                            off = np.arange(len(i)) - np.repeat(np.cumsum(cnt) - cnt, cnt)
                            j = order[np.repeat(start[k], cnt) + off]
                            if (a, b, z) == (0, 0, 0):
                                i, j = i[i < j], j[i < j]
                            yield i, j
        blocks = expand()
    for i, j in blocks:
        d = _image(pos[j] - pos[i], box)
        d2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
        ok = d2 < cut * cut
        yield i[ok], j[ok], d[ok], d2[ok]


def _pair_terms(kind, p, r):
    """(energy, F(r) / r with F along x_j - x_i on i) of a pair potential."""
    if kind == L.POT_HARMONIC_REPULSION:
        return 0.5 * p[0] * (r - p[1]) ** 2, p[0] * (r - p[1]) / r, p[1]
    if kind == L.POT_WEAK_INTERACTION:
        k, d0, h, rc = p
        c = (2.0 / (rc - d0)) ** 2
        near, mid = r < d0, r < d0 + 0.5 * (rc - d0)
        e = np.where(near, 0.5 * k * (r - d0) ** 2 - h,
                     np.where(mid, 0.5 * h * c * (r - d0) ** 2 - h, -0.5 * h * c * (r - rc) ** 2))
        f = np.where(near, -k * (d0 - r), np.where(mid, -h * c * (d0 - r), h * c * (rc - r)))
        return e, f / r, rc
    m, n, rc, shift, eps, sigma = p
    r_min = sigma * (n / m) ** (1.0 / (n - m))
    k = -eps / ((sigma / r_min) ** m - (sigma / r_min) ** n)
    q = sigma / r
    e = k * (q ** m - q ** n) - (k * ((sigma / rc) ** m - (sigma / rc) ** n) if shift else 0.0)
    return e, -k / sigma ** 2 * (m * q ** (m + 2) - n * q ** (n + 2)), rc


def _add(f, i, v):
    for a in range(3):
        f[:, a] += np.bincount(i, v[:, a], len(f))


def _bonded(pos, box, terms, f):
    """Harmonic bonds (100, 1), angles (10, pi) and cosine dihedrals (1, 3, 0) of the chains."""
    b, a, t = terms
    x = _image(pos[b[:, 1]] - pos[b[:, 0]], box)
    r = np.linalg.norm(x, axis=1)
    v = (200.0 * (r - 1.0) / r)[:, None] * x
    _add(f, b[:, 0], v)
    _add(f, b[:, 1], -v)
    energy = np.sum(100.0 * (r - 1.0) ** 2)
    u, w = _image(pos[a[:, 0]] - pos[a[:, 1]], box), _image(pos[a[:, 2]] - pos[a[:, 1]], box)
    u2, w2 = np.sum(u * u, 1), np.sum(w * w, 1)
    inv = 1.0 / np.sqrt(u2 * w2)
    ct = np.clip(np.sum(u * w, 1) * inv, -1.0, 1.0)
    theta = np.arccos(ct)
    c = 20.0 * (theta - np.pi) / np.maximum(np.sqrt(1.0 - ct * ct), 1e-10)
    gi = (c * ct / u2)[:, None] * u - (c * inv)[:, None] * w
    gk = (c * ct / w2)[:, None] * w - (c * inv)[:, None] * u
    _add(f, a[:, 0], -gi)
    _add(f, a[:, 1], gi + gk)
    _add(f, a[:, 2], -gk)
    energy += np.sum(10.0 * (theta - np.pi) ** 2)
    b1, b2 = _image(pos[t[:, 1]] - pos[t[:, 0]], box), _image(pos[t[:, 2]] - pos[t[:, 1]], box)
    b3 = _image(pos[t[:, 3]] - pos[t[:, 2]], box)
    # IUPAC angle psi of the torsion; the energy's angle is phi = -psi - pi
    A, B = np.cross(b1, b2), np.cross(b2, b3)
    n2 = np.linalg.norm(b2, axis=1)
    psi = np.arctan2(np.sum(np.cross(A, B) * b2, 1) / n2, np.sum(A * B, 1))
    phi = -psi - np.pi
    energy += np.sum(1.0 + np.cos(3.0 * phi))
    A2, B2 = np.sum(A * A, 1), np.sum(B * B, 1)
    cos_phi = np.cos(phi)
    dV = np.where(np.abs(cos_phi) < 1e-4, 0.0, -3.0 * np.sin(3.0 * phi))
    g1, g4 = -(n2 / A2)[:, None] * A, (n2 / B2)[:, None] * B
    p12, p32 = (np.sum(b1 * b2, 1) / n2 ** 2)[:, None], (np.sum(b3 * b2, 1) / n2 ** 2)[:, None]
    g2, g3 = -(1.0 + p12) * g1 + p32 * g4, p12 * g1 - (1.0 + p32) * g4
    for col, g in enumerate((g1, g2, g3, g4)):
        # the force is -dE/dx with dE/dphi = dV and dphi = -dpsi
        _add(f, t[:, col], dV[:, None] * g)
    return energy


class _Exact:
    """One system stepped in 64 bits."""

    def __init__(self, chem, box, pos, types, terms, seed):
        self.pots, self.rxs = chemistry(chem)
        self.D = np.array(DIFFUSION[chem])
        self.box, self.terms, self.seed = box, terms, seed
        self.pos, self.types = pos.copy(), types.astype(np.int64)
        self.handles = np.arange(len(types), dtype=np.int64)
        self.next = len(types)
        self.cut = max(p[1] if k == L.POT_HARMONIC_REPULSION else p[3] if k == L.POT_WEAK_INTERACTION else p[2]
                       for k, _, _, p in self.pots)
        self.reach = max(x.get("educt_distance", 0.0) for x in self.rxs)
        self.f, self.energy, self.step = None, 0.0, 0

    def forces(self):
        self.f, e = np.zeros_like(self.pos), 0.0
        for i, j, d, d2 in _pairs(self.pos, self.box, self.cut):
            r, ti, tj = np.sqrt(d2), self.types[i], self.types[j]
            for kind, a, b, p in self.pots:
                m = ((ti == a) & (tj == b)) | ((ti == b) & (tj == a))
                cut = _pair_terms(kind, p, np.ones(1))[2]
                m &= d2 < cut * cut
                en, fr, _ = _pair_terms(kind, p, r[m])
                e += en.sum()
                v = fr[:, None] * d[m]
                _add(self.f, i[m], v)
                _add(self.f, j[m], -v)
        if self.terms:
            e += _bonded(self.pos, self.box, self.terms, self.f)
        self.energy = e

    def integrate(self, dt):
        x = _philox(self.handles, self.step, 0, 0, self.seed)
        xi = _box_muller([((k >> np.uint64(8)).astype(float) + 0.5) * 2.0 ** -24 for k in x])
        D = self.D[self.types][:, None]
        self.pos = _wrap(self.pos + np.sqrt(2 * D * dt) * xi + self.f * D * dt, self.box)

    def react(self, handler, dt):
        events = []  # key, reaction, index of the first and second educt

        def accept(rx, k, a, b, x):
            u = _u53(x[0], x[1])
            if handler == "ua":
                key = (x[2] << np.uint64(32)) | x[3]
            else:
                key = -np.log(_u53(x[2], x[3]) + 2.0 ** -54) / rx["rate"]
            for m in np.nonzero(u < 1.0 - math.exp(-rx["rate"] * dt))[0]:
                events.append((key[m], k, int(a[m]), int(b[m])))

        near = list(_pairs(self.pos, self.box, self.reach)) if self.reach > 0 else []
        for k, rx in enumerate(self.rxs):
            ed = rx["educts"]
            if len(ed) == 1:
                a = np.nonzero(self.types == ed[0])[0]
                accept(rx, k, a, a, _philox(self.handles[a], self.step, 1 | (k << 8), 0, self.seed))
                continue
            for i, j, _, d2 in near:
                fwd = (self.types[i] == ed[0]) & (self.types[j] == ed[1])
                bwd = (self.types[i] == ed[1]) & (self.types[j] == ed[0])
                m = (fwd | bwd) & (d2 < rx["educt_distance"] ** 2)
                a, b = np.where(fwd, i, j)[m], np.where(fwd, j, i)[m]
                h1, h2 = self.handles[a], self.handles[b]
                accept(rx, k, a, b, _philox(np.minimum(h1, h2), self.step, 2 | (k << 8), np.maximum(h1, h2), self.seed))
        used, alive, born = set(), np.ones(len(self.pos), dtype=bool), []
        for _, k, a, b in sorted(events):
            if a in used or b in used:
                continue
            used.update((a, b))
            rx = self.rxs[k]
            if rx["kind"] == L.RX_ENZYMATIC:
                self.types[a], self.handles[a] = rx["products"][0], self.next
                self.next += 1
            elif rx["kind"] == L.RX_FUSION:
                alive[[a, b]] = False
                x = self.pos[a] + 0.5 * _image(self.pos[b] - self.pos[a], self.box)
                born.append((_wrap(x, self.box), rx["products"][0], self.next))
                self.next += 1
            else:
                alive[a] = False
                x = _philox(np.array([self.handles[a]]), self.step, 3, 0, self.seed)
                v = _box_muller([(w.astype(float) + 0.5) / 2.0 ** 32 for w in x])[0]
                v *= 0.5 * rx["product_distance"] / np.linalg.norm(v)
                born.append((_wrap(self.pos[a] - v, self.box), rx["products"][1], self.next))
                born.append((_wrap(self.pos[a] + v, self.box), rx["products"][0], self.next + 1))
                self.next += 2
        if born:
            x, t, h = zip(*born)
            self.pos = np.concatenate([self.pos[alive], np.array(x)])
            self.types = np.concatenate([self.types[alive], np.array(t, dtype=np.int64)])
            self.handles = np.concatenate([self.handles[alive], np.array(h, dtype=np.int64)])

    def loop(self, handler, dt, steps, every=None):
        """The steps; returns the species counts after every `every` steps and the energies of all."""
        counts, energies = [], []
        self.forces()
        for t in range(steps):
            self.integrate(dt)
            self.react(handler, dt)
            self.forces()
            self.step += 1
            energies.append(self.energy)
            if every and ((t + 1) % every == 0 or t + 1 == steps):
                counts.append(np.bincount(self.types, minlength=3))
        return np.array(counts, dtype=np.int64), np.array(energies)

    def particles(self):
        o = np.argsort(self.handles)
        return self.pos[o], self.types[o], self.handles[o]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("ensemble", "serve"):
        reps = _replicas(case, seed)
        if sum(n * steps for n, _, _, _, steps in reps) * (1.0 + 10.0 * case["density"]) > 8e6:
            return None
        parts, tables = [], []
        for n, box, sd, handler, steps in reps:
            s = _Exact(case["chem"], box, *_replica_state(n, box, sd), None, sd)
            tables.append(s.loop(handler, case["dt"], steps, case.get("interval", steps))[0])
            parts.append(s.particles())
        rows = sum(_rows(rep[0]) for rep in reps)
        return dict(_frame(parts, rows), counts=np.concatenate(tables) if kind == "ensemble" else None)
    cost = case["n"] * case.get("steps", 1) * (1.0 + 10.0 * case["density"])
    if cost > (8e6 if kind in ("run", "actions") else 6e6):
        return None
    pos, types, terms, box = _system(case, seed)
    if kind == "rdf":
        if case["n"] * case["density"] * case["r_max"] ** 3 > 2e6:
            return None
        borders, hist = np.linspace(0.0, case["r_max"], case["bins"] + 1), np.zeros(case["bins"] + 2, dtype=np.int64)
        for _, _, _, d2 in _pairs(pos, box, case["r_max"] * (1.0 + 1e-9)):
            hist += 2 * np.bincount(np.searchsorted(borders, np.sqrt(d2), side="right"), minlength=case["bins"] + 2)
        return {"counts": hist[1:-1], "n_from": case["n"]}
    s = _Exact(case["chem"], box, pos, types, terms, seed)
    if kind == "forces":
        s.forces()
        return {"forces": s.f, "handles": s.handles, "energy": float(s.energy)}
    counts, energies = s.loop(case["handler"], case["dt"], case["steps"], case.get("every"))
    out = _frame([s.particles()], _rows(case["n"]))
    return dict(out, counts=counts) if kind == "run" else dict(out, energies=energies)
