"""DVND rounds that leave out blocks of moves which cannot improve
(csrc/mlp_prune.h) against the oracle, which evaluates every move: tours,
latencies, round counts and the rows that can be read afterwards.

Sizes around the 16-position blocks, the eight rows of a wave and the columns
of a wave; start tours whose 2-opt deltas need 64 bits, and coordinates that
take swap and or-opt deltas beyond 32 bits.  Whole numbers: no tolerance.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

wm = pytest.importorskip("wamca_mi")


@pytest.fixture(scope="module")
def eng():
    e = wm.Engine(0)
    yield e
    e.close()


def _rows_equal(eng, s, nb, ref):
    got = eng.rows(s, nb)
    return all(np.array_equal(got[k], ref[k]) for k in ("cost", "i", "j"))


@pytest.mark.parametrize("rnd", [0, 1])
@pytest.mark.parametrize("sizes", [(2, 3, 4, 5, 6, 7, 8, 9, 260), (14, 15, 16, 17, 23, 31, 32, 33, 271, 255),
                                   (47, 64, 126, 127, 128, 129, 256, 257, 272), (511,), (513,), (1023, 1024)])
def test_dvnd_and_rows_after(eng, sizes, rnd):
    """One call over slots of these sizes (the largest decides that rounds are
    pruned)."""
    insts, slots, tours, Ws = [], [], [], []
    for q, n in enumerate(sizes):
        xs, ys = (O.instance_clustered if n % 2 else O.instance_uniform)(n, 40 + n)
        Ws.append(O.weights(xs, ys, rnd))
        tours.append(O.random_tour(O.MT(n), Ws[q], 0.5))
        insts.append(eng.instance(xs, ys, rnd))
        slots.append(eng.slot(insts[q]))
    try:
        eng.set_tours(slots, tours)
        rounds = eng.dvnd(slots)
        lat = eng.latency(slots)
        for q, s in enumerate(slots):
            tref, Lref, rref, _ = O.dvnd(Ws[q], tours[q], 0)
            assert (int(lat[q]), int(rounds[q])) == (Lref, rref), sizes[q]
            assert np.array_equal(eng.get_tour(s), tref), sizes[q]
            # the last round applied nothing: its rows are the final tour's
            for nb in range(5):
                if O.rows(nb, 0, len(tref)) > 0 and len(tref) > 5:
                    assert _rows_equal(eng, s, nb, O.eval_rows(nb, 0, Ws[q], tref)), (sizes[q], nb)
    finally:
        for s in slots:
            eng.destroy_slot(s)
        for i in insts:
            eng.destroy_instance(i)


@pytest.mark.parametrize("max_rounds", [1, 2, 5, 6])
def test_rows_after_max_rounds(eng, max_rounds):
    """Rows read after a run that max_rounds ended are those of its last round,
    each neighborhood's before its merge."""
    sizes = (90, 300)
    insts, slots, tours, Ws = [], [], [], []
    for q, n in enumerate(sizes):
        xs, ys = O.instance_uniform(n, 7 + q)
        Ws.append(O.weights(xs, ys, 1))
        tours.append(O.random_tour(O.MT(q + 1), Ws[q], 0.5))
        insts.append(eng.instance(xs, ys, 1))
        slots.append(eng.slot(insts[q]))
    try:
        eng.set_tours(slots, tours)
        rounds = eng.dvnd(slots, 0, max_rounds)
        for q, s in enumerate(slots):
            t = tours[q]
            for r in range(int(rounds[q])):
                refs = []
                for nb in range(5):
                    refs.append(O.eval_rows(nb, 0, Ws[q], t))
                    t = O.step(nb, 0, Ws[q], t)[0]
            assert np.array_equal(eng.get_tour(s), t)
            for nb in range(5):
                assert _rows_equal(eng, s, nb, refs[nb]), (q, nb)
    finally:
        for s in slots:
            eng.destroy_slot(s)
        for i in insts:
            eng.destroy_instance(i)


@pytest.mark.parametrize("n,span,max_rounds", [(1024, 1000, 0), (2300, 1000, 8), (6001, 32767, 2)])
def test_wide_deltas(eng, n, span, max_rounds):
    """n = 2300: 2-opt deltas of the first rounds beyond 32 bits; n = 6001 with
    coordinates up to 32767: swap and or-opt deltas too."""
    xs, ys = O.instance_uniform(n, 5, span)
    t0 = O.perm_tour(3, n)
    inst = eng.instance(xs, ys, 1)
    s = eng.slot(inst)
    try:
        eng.set_tour(s, t0)
        rounds = int(eng.dvnd([s], 0, max_rounds)[0])
        tref, Lref, rref = O.dvnd_xy(xs, ys, 1, t0, 0, max_rounds)[:3]
        assert (int(eng.latency([s])[0]), rounds) == (Lref, rref)
        assert np.array_equal(eng.get_tour(s), tref)
    finally:
        eng.destroy_slot(s)
        eng.destroy_instance(inst)
