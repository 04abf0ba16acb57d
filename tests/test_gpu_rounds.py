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
