"""The work that is timed: what programs have this library do, over its range.

A case is one of six kinds of call:

``static``  every neighborhood of one tour in device memory, through the entry
            point that allocates nothing (a caller's own search loop asking
            for the best move of each row);
``evals``   every neighborhood of several tours in one launch, each row's best
            move as a 64-bit record in device memory;
``dvnd``    set tours, run DVND, read the tours, latencies and round counts
            (one solve, or a batch of unequal instances in one call);
``round``   the same for many tours of one instance and a limited number of
            rounds (a population's local-search step);
``served``  a list of jobs handed to the continuous-batching server at once;
``total``   TOTAL mode: every thread slot's best move, its merge and the moves
            it applied.

Sizes are those of the benchmark, the tests and the instance files in
tests/golden, and odd ones between them.  Inputs come from the library's own
seeded generators, as in its benchmark: uniform coordinates in [0, 1000]^2 or
20 Gaussian clusters in [0, 2000]^2, random permutations and tours of the
randomized construction; and tours along strips of the plane.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "wamca-gpu-mi_amd"))

import wamca_mi  # noqa: E402
from wamca_mi import inputs, serve  # noqa: E402

ALL = 0x1F  # swap, 2-opt, or-opt-1/2/3
ADS, ODC = 0, 1

_eng = None


def engine():
    """The context that a program keeps for all of its calls."""
    global _eng
    if _eng is None:
        _eng = wamca_mi.Engine(0)
    return _eng


def listed():
    return [
        # one small tour's neighborhoods: launches and their latency
        {"name": "static_n100", "kind": "static", "n": 100, "rowmap": ADS, "tour": "perm"},
        # the headline: n = 1000, one tour per call, row map of the ADS kernels
        {"name": "static_n1000", "kind": "static", "n": 1000, "rowmap": ADS, "tour": "perm"},
        # the same under the row map of the drop-in surfaces
        {"name": "static_n1000_odc", "kind": "static", "n": 1000, "rowmap": ODC, "tour": "perm"},
        # a long random tour: 2-opt deltas beyond 32 bits
        {"name": "static_n3001", "kind": "static", "n": 3001, "rowmap": ADS, "tour": "perm"},
        # eight long tours of short edges in one launch (a search in its later stages)
        {"name": "evals_8x4001", "kind": "evals", "n": 4001, "count": 8, "rowmap": ADS, "tour": "near"},
        # one round over a population of start tours
        {"name": "round_256x784", "kind": "round", "n": 784, "count": 256, "rounds": 1, "rowmap": ADS},
        # a small solve alone
        {"name": "dvnd_n100", "kind": "dvnd", "count": 1, "lo": 100, "hi": 100, "clustered": False, "rowmap": ADS},
        # an ordinary solve alone
        {"name": "dvnd_n1000", "kind": "dvnd", "count": 1, "lo": 1000, "hi": 1000, "clustered": False, "rowmap": ADS},
        # 64 unequal instances in one call
        {"name": "dvnd_64", "kind": "dvnd", "count": 64, "lo": 50, "hi": 2000, "sizes": 3, "rowmap": ADS},
        # a large clustered solve, beyond the merge that fits in LDS
        {"name": "dvnd_n9001", "kind": "dvnd", "count": 1, "lo": 9001, "hi": 9001, "clustered": True, "rowmap": ADS},
        # a burst of jobs at the server
        {"name": "served_100", "kind": "served", "count": 100, "lo": 100, "hi": 1000, "sizes": 3},
        # the reference's TOTAL experiment at its largest logged size
        {"name": "total_n1000", "kind": "total", "n": 1000, "nb": 2, "block": 896},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["static", "static", "static", "evals", "round", "dvnd", "dvnd", "dvnd", "served", "total"])
    if kind == "static":
        return {"kind": kind, "n": _log(rng, 50, 3001), "rowmap": rng.choice([ADS, ODC]), "tour": rng.choice(["perm", "near"])}
    if kind == "evals":
        n = _log(rng, 200, 4001)
        return {"kind": kind, "n": n, "count": rng.randint(2, max(2, min(32, int(8 * 4001 * 4001 / (n * n))))),
                "rowmap": ADS, "tour": "near"}
    if kind == "round":
        n = _log(rng, 100, 1000)
        return {"kind": kind, "n": n, "count": rng.randint(16, max(16, min(256, int(256 * 784 * 784 / (n * n))))),
                "rounds": rng.randint(1, 2) if n < 500 else 1, "rowmap": ADS}
    if kind == "dvnd":
        if rng.random() < 0.5:
            n = _log(rng, 50, 7000)
            return {"kind": kind, "count": 1, "lo": n, "hi": n, "clustered": rng.random() < 0.5,
                    "rowmap": ADS if n > 1000 else rng.choice([ADS, ADS, ODC])}
        return {"kind": kind, "count": rng.randint(2, 64), "lo": 50, "hi": _log(rng, 100, 2000),
                "sizes": rng.randint(1, 1000), "rowmap": ADS}
    if kind == "served":
        return {"kind": kind, "count": rng.randint(8, 100), "lo": 100, "hi": _log(rng, 200, 1000), "sizes": rng.randint(1, 1000)}
    return {"kind": kind, "n": _log(rng, 100, 1000), "nb": rng.randint(0, 4), "block": rng.choice([64, 128, 576, 896])}


class State:
    """What a program holds between calls; its slots and instances go back to
    the context with it."""

    def __init__(self, case):
        self.kind = case["kind"]
        self.insts, self.slots = [], []

    def __del__(self):
        try:
            for s in self.slots:
                _eng.destroy_slot(s)
            for i in self.insts:
                _eng.destroy_instance(i)
        except Exception:
            pass


def _coords(n, seed, clustered):
    return inputs.clustered(n, seed) if clustered else inputs.uniform(n, seed, 1000)


def _tour(how, xs, ys, seed):
    if how == "perm":
        return inputs.perm_tour(seed, len(xs))
    # up and down strips of the plane, of random width and slightly shuffled:
    # edges about as short as after a constructive heuristic
    n = len(xs)
    rng = np.random.RandomState(seed % 2**31)
    width = math.sqrt(3e6 / n) * rng.uniform(0.8, 1.25)
    strip = (xs / width).astype(np.int64)
    y = ys + rng.normal(0.0, 0.2 * width, n)
    order = np.lexsort((np.where(strip % 2 == 0, y, -y), strip))
    return np.concatenate([[0], order[order != 0], [0]]).astype(np.int32)


def _jobs(case, seed):
    """Instances and start tours as in the package's job streams: sizes
    log-uniform in [lo, hi], half uniform, half clustered."""
    jobs = []
    for q in range(case["count"]):
        n = inputs.loguniform_n(case["sizes"], q, case["lo"], case["hi"])
        xs, ys = _coords(n, seed + q, q % 2 == 1)
        jobs.append((xs, ys, inputs.random_tour(xs, ys, 1, seed + q)))
    return jobs


def _rows(n, rowmap):
    return [wamca_mi.rows_of(nb, rowmap, n + 1) for nb in range(5)]


def prepare(case, seed):
    eng = engine()
    st = State(case)
    kind = case["kind"]
    seed = seed * 7919 + 1
    if kind == "served" or (kind == "dvnd" and case["count"] > 1):
        jobs = _jobs(case, seed)
        if kind == "served":
            st.jobs = jobs
            return st
        for xs, ys, _ in jobs:
            st.insts.append(eng.instance(xs, ys, 1))
            st.slots.append(eng.slot(st.insts[-1]))
        st.tours = [t for _, _, t in jobs]
        st.rowmap, st.rounds = case["rowmap"], 0
        return st
    n = case["lo"] if kind == "dvnd" else case["n"]
    xs, ys = _coords(n, seed, kind == "round" or case.get("clustered", False))
    st.insts.append(eng.instance(xs, ys, 1))
    if kind == "dvnd":
        st.slots.append(eng.slot(st.insts[0]))
        make = inputs.random_tour_fast if n > 4000 else inputs.random_tour
        st.tours = [make(xs, ys, 1, seed)]
        st.rowmap, st.rounds = case["rowmap"], 0
    elif kind == "round":
        st.slots = eng.slots(st.insts[0], case["count"])
        st.tours = [inputs.perm_tour(seed + q, n) for q in range(case["count"])]
        st.rowmap, st.rounds = case["rowmap"], case["rounds"]
    elif kind == "static":
        st.rowmap = case["rowmap"]
        rows = sum(_rows(n, st.rowmap))
        st.tour = torch.from_numpy(_tour(case["tour"], xs, ys, seed)).cuda()
        st.cost = torch.empty(rows, dtype=torch.int64, device="cuda")
        st.i = torch.empty(rows, dtype=torch.int32, device="cuda")
        st.j = torch.empty(rows, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()  # the tour is there before the context's stream reads it
    elif kind == "evals":
        st.rowmap = case["rowmap"]
        st.slots = eng.slots(st.insts[0], case["count"])
        eng.set_tours(st.slots, [_tour(case["tour"], xs, ys, seed + q) for q in range(case["count"])])
        st.rows = _rows(n, st.rowmap)
        st.moves = torch.empty((case["count"], sum(st.rows)), dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
    else:
        st.slots.append(eng.slot(st.insts[0]))
        st.tours = [_tour("perm", xs, ys, seed)]
        st.nb, st.block = case["nb"], case["block"]
    return st


def run(st):
    eng = engine()
    if st.kind == "static":
        eng._ck(eng._L.mlp_eval_static(eng.h, st.insts[0], st.tour.data_ptr(), ALL, st.rowmap, st.cost.data_ptr(),
                                       st.i.data_ptr(), st.j.data_ptr()))
        return {"cost": st.cost, "i": st.i, "j": st.j}
    if st.kind == "evals":
        eng.eval(st.slots, ALL, st.rowmap)
        moves64 = eng._L.mlp_rows_moves64_device
        count = ctypes.c_int32()
        at = st.moves.data_ptr()
        for s in st.slots:
            for nb, rows in enumerate(st.rows):
                eng._ck(moves64(eng.h, s, nb, ctypes.c_void_p(at), ctypes.c_int64(rows), ctypes.byref(count)))
                at += 8 * rows
        return st.moves
    if st.kind == "served":
        out = serve.run_served(eng, st.jobs, [0.0] * len(st.jobs))
        return {"latency": np.array(out["latency"], np.int64), "rounds": np.array(out["rounds"], np.int32),
                "tours": np.concatenate(out["tours"])}
    if st.kind == "total":
        eng.set_tours(st.slots, st.tours)
        eng.eval_total(st.slots, st.nb, st.block)
        entries = eng.total(st.slots[0])
        eng.merge_total(st.slots)
        applied = np.array(eng.applied(st.slots[0], st.nb), np.int64).reshape(-1, 5)
        # as many rows as there can be: the count of kept moves differs from tour to tour
        applied = np.concatenate([applied, np.zeros((len(st.tours[0]) - len(applied), 5), np.int64)])
        return {"entries": entries, "applied": applied,
                "latency": eng.latency(st.slots), "tours": np.concatenate(eng.get_tours(st.slots))}
    eng.set_tours(st.slots, st.tours)
    rounds = eng.dvnd(st.slots, st.rowmap, st.rounds)
    return {"latency": eng.latency(st.slots), "rounds": rounds, "tours": np.concatenate(eng.get_tours(st.slots))}


def _moves(n):
    N = n + 1
    return (N - 4) * (N - 3) // 2 + (N - 2) * (N - 3) // 2 + sum((N - k - 2) * (N - k - 1) for k in (1, 2, 3))


def work(case):
    """Ten integer operations a move.  A DVND solve cannot do without one
    evaluation of every neighborhood of its result (that it is a local optimum),
    a round not without one of its start."""
    kind = case["kind"]
    if kind in ("served", "dvnd"):
        lo, hi = case["lo"], case["hi"]
        if lo == hi:
            n1, n2 = lo, _moves(lo)
        else:  # means over n log-uniform in [lo, hi]
            w = math.log(hi / lo)
            n1, n2 = (hi - lo) / w, 4 * (hi * hi - lo * lo) / 2 / w
        return {"bytes": case["count"] * (8 * n1 + 8 * n1 + 20), "flops": case["count"] * 10 * n2}
    n = case["n"]
    if kind == "round":
        return {"bytes": 8 * n + case["count"] * (8 * n + 12), "flops": case["count"] * case["rounds"] * 10 * _moves(n)}
    if kind == "static":
        return {"bytes": 12 * n + 16 * sum(_rows(n, case["rowmap"])), "flops": 10 * _moves(n)}
    if kind == "evals":
        return {"bytes": 8 * n + case["count"] * (4 * n + 8 * sum(_rows(n, ADS))), "flops": 10 * case["count"] * _moves(n)}
    rows = wamca_mi.rows_of(case["nb"], ADS, n + 1)
    return {"bytes": 16 * n + 16 * rows * case["block"], "flops": 10 * _moves(n) / 4}


def _grid(nb, rowmap, N, r):
    """i and j of every row-local index of rows r (a column), and where they are moves."""
    if nb == 0:
        c = np.arange(N - 1 if rowmap == ADS else N - 4)[None, :]
        if rowmap == ADS:
            return r + 1 + 0 * c, c + 0 * r, c >= r + 3
        up = c >= r
        return np.where(up, r + 1, N - r - 3), np.where(up, c + 3, N - c - 2), up | ~up
    if nb == 1:
        c = np.arange(N - 3)[None, :]
        up = c >= r
        return np.where(up, c - r + 1, r - c), np.where(up, c + 2, N - c - 2), up | ~up
    k = nb - 1
    if rowmap == ADS:
        c = np.arange(N - k - 1)[None, :]
        return np.where(c > r, r + 1, r + 2) + 0 * c, c + 1 + 0 * r, (c >= 0) | (r < 0)
    c = np.arange(N - k - 2)[None, :]
    up = c >= r
    return np.where(up, c - r + 1, N - c - k - 1), np.where(up, c + 2, r - c), up | ~up


def _deltas(nb, i, j, x, y, T, Q):
    """Change of the tour's latency (the sum of the arrival times) by a move,
    from rounded Euclidean distances and the prefix sums T of the edges and Q
    of position times edge."""
    N = len(x)

    def d(a, b):
        s = (x[a] - x[b]) ** 2 + (y[a] - y[b]) ** 2
        return np.floor(np.sqrt(s.astype(np.float64)) + 0.5).astype(np.int64)

    def w(p):
        return T[p] - T[p - 1]

    if nb == 0:
        return ((N - i) * (d(i - 1, j) - w(i)) + (N - i - 1) * (d(j, i + 1) - w(i + 1)) +
                (N - j) * (d(j - 1, i) - w(j)) + (N - j - 1) * (d(i, j + 1) - w(j + 1)))
    if nb == 1:
        return ((N - i) * (d(i - 1, j) - w(i)) + (N - j - 1) * (d(i, j + 1) - w(j + 1)) +
                2 * (Q[j] - Q[i]) - (i + j + 1) * (T[j] - T[i]))
    k = nb - 1
    seg = T[i + k - 1] - T[i]
    jf = np.maximum(i + 1, j)  # the segment moves towards the end
    f = ((N - i) * (d(i - 1, np.minimum(i + k, N - 1)) - w(i)) + (N - jf - k) * (d(i + k - 1, np.minimum(jf + k, N - 1)) - w(np.minimum(jf + k, N - 1))) +
         (N - jf) * d(np.minimum(jf + k - 1, N - 1), i) - (N - i - k) * w(np.minimum(i + k, N - 1)) +
         (i - jf) * seg + k * (T[np.minimum(jf + k - 1, N - 1)] - T[np.minimum(i + k, N - 1)]))
    jb = np.minimum(i - 1, j)  # towards the start
    b = ((N - jb) * (d(jb - 1, i) - w(jb)) + (N - i - k) * (d(i - 1, i + k) - w(i + k)) +
         (N - jb - k) * d(i + k - 1, jb) - (N - i) * w(i) + (i - jb) * seg - k * (T[i - 1] - T[jb]))
    return np.where(i < j, f, b)


def exact(case, seed):
    """Each row's best move of a ``static`` case in 64-bit numpy; the other
    kinds return tours and moves of a search, which have no value of their own."""
    if case["kind"] != "static":
        return None
    n = case["n"]
    seed = seed * 7919 + 1
    xs, ys = _coords(n, seed, False)
    t = _tour(case["tour"], xs, ys, seed)
    N = n + 1
    x, y = xs[t].astype(np.int64), ys[t].astype(np.int64)
    s = (x[1:] - x[:-1]) ** 2 + (y[1:] - y[:-1]) ** 2
    w = np.concatenate([[0], np.floor(np.sqrt(s.astype(np.float64)) + 0.5).astype(np.int64)])
    T, Q = np.cumsum(w), np.cumsum(np.arange(N) * w)
    out = {"cost": [], "i": [], "j": []}
    for nb, rows in enumerate(_rows(n, case["rowmap"])):
        for r0 in range(0, rows, 128):
            r = np.arange(r0, min(rows, r0 + 128))[:, None]
            i, j, ok = _grid(nb, case["rowmap"], N, r)
            # indices that are no moves are evaluated in place of a valid one
            v = np.where(ok, _deltas(nb, np.where(ok, i, 1), np.where(ok, j, 3), x, y, T, Q), np.iinfo(np.int64).max)
            at = v.argmin(axis=1)[:, None]  # the first of equal ones: the lowest index
            for name, a in (("cost", v), ("i", i), ("j", j)):
                out[name].append(np.take_along_axis(np.broadcast_to(a, v.shape), at, axis=1)[:, 0])
    return {"cost": np.concatenate(out["cost"]), "i": np.concatenate(out["i"]).astype(np.int32),
            "j": np.concatenate(out["j"]).astype(np.int32)}
