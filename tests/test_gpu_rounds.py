"""mlp_dvnd calls repeated on the same slots, whose chunks of rounds replay
recorded graphs from the third call on (tests/test_dvnd_host.py counts them):
every call against the oracle, with new tours each time and the program's own
evaluations between the calls.  Whole numbers: no tolerance.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

wm = pytest.importorskip("wamca_mi")
from wamca_mi import inputs  # noqa: E402


@pytest.fixture(scope="module")
def eng():
    e = wm.Engine(0)
    yield e
    e.close()


def _rows_equal(eng, s, nb, ref):
    got = eng.rows(s, nb)
    return all(np.array_equal(got[k], ref[k]) for k in ("cost", "i", "j"))


@pytest.mark.parametrize("rowmap", [0, 1])
@pytest.mark.parametrize("max_rounds", [3, 5, 8, 9])
def test_repeated_limited_calls(eng, max_rounds, rowmap):
    sizes = (90, 300)
    insts, slots, Ws = [], [], []
    for q, n in enumerate(sizes):
        xs, ys = O.instance_uniform(n, 70 + q)
        Ws.append(O.weights(xs, ys, 1))
        insts.append(eng.instance(xs, ys, 1))
        slots.append(eng.slot(insts[q]))
    try:
        for call in range(5):
            tours = [O.random_tour(O.MT(10 * call + q + 1), W, 0.5) for q, W in enumerate(Ws)]
            eng.set_tours(slots, tours)
            rounds = eng.dvnd(slots, rowmap, max_rounds)
            for q, s in enumerate(slots):
                t = tours[q]
                for _ in range(int(rounds[q])):
                    refs = []
                    for nb in range(5):
                        refs.append(O.eval_rows(nb, rowmap, Ws[q], t))
                        t = O.step(nb, rowmap, Ws[q], t)[0]
                assert int(rounds[q]) == max_rounds or np.array_equal(t, O.dvnd(Ws[q], tours[q], rowmap)[0])
                assert np.array_equal(eng.get_tour(s), t), (call, q)
                for nb in range(5):
                    assert _rows_equal(eng, s, nb, refs[nb]), (call, q, nb)
            eng.eval(slots, 0x1F, 1 - rowmap)
    finally:
        for s in slots:
            eng.destroy_slot(s)
        for i in insts:
            eng.destroy_instance(i)


@pytest.mark.parametrize("n,rnd", [(2500, 1), (6001, 0)])
def test_wide_rows_completed(eng, n, rnd):
    """A run that stops in a round which left rows out, on a tour whose deltas
    need 64 bits there: 2-opt at n = 2500, swap and or-opt too at n = 6001
    (coordinates up to 32767).  The rows are completed after the run."""
    xs, ys = O.instance_uniform(n, 9, 32767)
    inst = eng.instance(xs, ys, rnd)
    s = eng.slot(inst)
    try:
        eng.set_tour(s, O.perm_tour(3, n) if n < 4000 else inputs.random_tour_fast(xs, ys, rnd, 3))
        eng.dvnd([s])
        t0 = eng.get_tour(s)
        T = int(O.latency_xy(xs, ys, rnd, t0)) // n  # below the tour's length
        md = 46342  # the bounds of the 32-bit paths
        assert (n + 1) * (T + 6 * md) + 3 * T >= 2**31 and (n < 4000 or 8 * (n + 1) * md >= 2**31)
        t0[n // 2:n // 2 + 8] = t0[n // 2:n // 2 + 8][::-1].copy()
        t0[n // 3:n // 3 + 5] = np.roll(t0[n // 3:n // 3 + 5], 2)
        for _ in range(2):
            eng.set_tour(s, t0)
            rounds = int(eng.dvnd([s])[0])
            tref, Lref, rref = O.dvnd_xy(xs, ys, rnd, t0, 0)[:3]
            assert rref > 1
            assert (int(eng.latency([s])[0]), rounds) == (Lref, rref)
            assert np.array_equal(eng.get_tour(s), tref)
            for nb in range(5):
                got, ref = eng.rows(s, nb), O.eval_rows_xy(nb, 0, xs, ys, rnd, tref)
                assert all(np.array_equal(got[k], ref[k]) for k in ("cost", "i", "j")), nb
    finally:
        eng.destroy_slot(s)
        eng.destroy_instance(inst)
