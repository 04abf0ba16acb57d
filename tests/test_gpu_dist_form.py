"""Launches whose slots all have short distances (every squared distance below
2^21) use the shorter distance form, others the general one: rows against the
oracle where the choice can go wrong - both sides of the limit, launches of both
kinds of slots, and recorded launches (a caller's graph, a DVND chunk's) replayed
after a slot was made again from an instance of the other kind.  Whole numbers:
no tolerance.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

wm = pytest.importorskip("wamca_mi")

ALL = 0x1F


@pytest.fixture(scope="module")
def eng():
    e = wm.Engine(0)
    yield e
    e.close()


def _inst(n, span, seed):
    """Coordinates over [0, span]^2 with both corners."""
    rng = np.random.RandomState(seed)
    xs, ys = rng.randint(0, span + 1, (2, n)).astype(np.int32)
    xs[1], ys[1], xs[2], ys[2] = 0, 0, span, span
    return xs, ys


def _rows_equal(eng, s, rowmap, xs, ys, rnd, tour):
    for nb in range(5):
        got, ref = eng.rows(s, nb), O.eval_rows_xy(nb, rowmap, xs, ys, rnd, tour)
        assert all(np.array_equal(got[k], ref[k]) for k in ("cost", "i", "j")), nb


@pytest.mark.parametrize("tile", [-1, 0, 1, 2, 3, 4])
@pytest.mark.parametrize("rnd", [0, 1])
@pytest.mark.parametrize("spans", [(1000,), (1023,), (1024,), (1025,), (32767,), (1000, 32767), (1024, 1000, 1025)])
def test_rows(eng, spans, rnd, tile):
    """span 1024: the diagonal is 1448.2, the largest that counts as short."""
    n = 301
    data = [_inst(n, span, 7 * q + span) for q, span in enumerate(spans)]
    insts = [eng.instance(x, y, rnd) for x, y in data]
    slots = [eng.slot(i) for i in insts]
    tours = [O.perm_tour(q + 1, n) for q in range(len(spans))]
    eng.set_tile(tile)
    try:
        eng.set_tours(slots, tours)
        for rowmap in (0, 1):
            eng.eval(slots, ALL, rowmap)
            for s, (xs, ys), t in zip(slots, data, tours):
                _rows_equal(eng, s, rowmap, xs, ys, rnd, t)
    finally:
        eng.set_tile(-1)
        for s in slots:
            eng.destroy_slot(s)
        for i in insts:
            eng.destroy_instance(i)


@pytest.mark.parametrize("rowmap", [0, 1])
@pytest.mark.parametrize("first,second", [(1000, 32767), (32767, 1000)])
def test_graph_after_slot_made_again(eng, first, second, rowmap):
    n, rnd = 130, 1
    inst = eng.instance(*_inst(n, first, 1), rnd)
    s = eng.slot(inst)
    tour = O.perm_tour(5, n)
    eng.set_tour(s, tour)
    eng.eval([s], ALL, rowmap)
    eng.sync()
    eng.graph_begin()
    eng.eval([s], ALL, rowmap)
    g = eng.graph_end()
    try:
        for k, span in enumerate((first, second, first)):
            if k:
                eng.destroy_slot(s)
                eng.destroy_instance(inst)
                inst = eng.instance(*_inst(n, span, 1), rnd)
                assert eng.slot(inst) == s
                eng.set_tour(s, tour)
            xs, ys = _inst(n, span, 1)
            for _ in range(3):
                eng.graph_launch(g)
                _rows_equal(eng, s, rowmap, xs, ys, rnd, tour)
    finally:
        eng.graph_destroy(g)
        eng.destroy_slot(s)
        eng.destroy_instance(inst)


@pytest.mark.parametrize("rowmap", [0, 1])
@pytest.mark.parametrize("n", [130, 300])
@pytest.mark.parametrize("first,second", [(1000, 32767), (32767, 1000)])
def test_dvnd_after_slot_made_again(eng, first, second, n, rowmap):
    """Three calls on each instance: the chunks' graphs are recorded."""
    rnd, s, inst = 1, None, None
    tour = O.perm_tour(5, n)
    try:
        for span in (first, second, first):
            if s is not None:
                eng.destroy_slot(s)
                eng.destroy_instance(inst)
            xs, ys = _inst(n, span, 2)
            inst = eng.instance(xs, ys, rnd)
            s2 = eng.slot(inst)
            assert s is None or s2 == s
            s = s2
            ref = O.dvnd_xy(xs, ys, rnd, tour, rowmap)
            for _ in range(3):
                eng.set_tour(s, tour)
                rounds = int(eng.dvnd([s], rowmap)[0])
                assert (int(eng.latency([s])[0]), rounds) == (ref[1], ref[2]), span
                assert np.array_equal(eng.get_tour(s), ref[0]), span
                _rows_equal(eng, s, rowmap, xs, ys, rnd, ref[0])
    finally:
        eng.destroy_slot(s)
        eng.destroy_instance(inst)
