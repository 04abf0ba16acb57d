"""Merges over more slots than the GPU has CUs, which take narrower workgroups
(csrc/mlp_kernels.hip MLP_MERGE_FOR) and read one row buffer only, against the
oracle's serial greedy: the kept moves in their order, the tour, the latency;
and the same inside DVND rounds, with slots that stop before the others.

The largest tour of a launch decides its workgroup: sizes on both sides of each
limit.  Whole numbers: no tolerance.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

wm = pytest.importorskip("wamca_mi")

SMALL = 280  # slots beside the large ones


@pytest.fixture(scope="module")
def eng():
    e = wm.Engine(0)
    yield e
    e.close()


def _slots(eng, large):
    ns = [20 + q % 60 for q in range(SMALL)] + list(large)
    xys = [(O.instance_clustered if q % 2 else O.instance_uniform)(n, 900 + q) for q, n in enumerate(ns)]
    insts = [eng.instance(x, y, 1) for x, y in xys]
    return ns, xys, insts, [eng.slot(i) for i in insts]


def _release(eng, insts, slots):
    for s in slots:
        eng.destroy_slot(s)
    for i in insts:
        eng.destroy_instance(i)


@pytest.mark.parametrize("rowmap", [0, 1])
@pytest.mark.parametrize("large", [(90,), (255, 100), (256, 300), (511,), (512, 513), (1022, 1023), (1024, 1026),
                                   (2047, 600), (2048, 2050)])
def test_merges(eng, large, rowmap):
    ns, xys, insts, slots = _slots(eng, large)
    try:
        tours = [O.perm_tour(q + 1, n) for q, n in enumerate(ns)]
        looked = list(range(0, SMALL, 40)) + list(range(SMALL, len(ns)))
        for nb in (0, 1, 3):
            eng.set_tours(slots, tours)
            for _ in range(2):  # both row buffers
                eng.eval(slots, 1 << nb, rowmap)
            eng.merge_apply(slots, nb)
            for q in looked:
                (xs, ys), t = xys[q], tours[q]
                ref = O.eval_rows_xy(nb, rowmap, xs, ys, 1, t)
                kept, _ = O.merge(nb, ref["cost"], ref["i"], ref["j"])
                want = [(int(ref["cost"][r]), nb, int(ref["i"][r]), int(ref["j"][r]), int(r)) for r in kept]
                for _, _, i, j, _ in want:
                    t = O.apply(nb, t, i, j)
                assert eng.applied(slots[q], nb) == want, (nb, ns[q])
                assert np.array_equal(eng.get_tour(slots[q]), t), (nb, ns[q])
                assert int(eng.latency([slots[q]])[0]) == O.latency_xy(xs, ys, 1, t), (nb, ns[q])
    finally:
        _release(eng, insts, slots)


@pytest.mark.parametrize("rowmap", [0, 1])
@pytest.mark.parametrize("large", [(60,), (300, 700), (1500,)])
def test_dvnd(eng, large, rowmap):
    ns, xys, insts, slots = _slots(eng, large)
    eng.dvnd_groups(1)
    try:
        tours = [O.perm_tour(q + 1, n) for q, n in enumerate(ns)]
        eng.set_tours(slots, tours)
        rounds = eng.dvnd(slots, rowmap, 12)
        lat = eng.latency(slots)
        got = eng.get_tours(slots)
        for q in list(range(0, SMALL, 20)) + list(range(SMALL, len(ns))):
            tref, Lref, rref = O.dvnd_xy(xys[q][0], xys[q][1], 1, tours[q], rowmap, 12)[:3]
            assert (int(lat[q]), int(rounds[q])) == (Lref, rref), ns[q]
            assert np.array_equal(got[q], tref), ns[q]
    finally:
        eng.dvnd_groups(2)
        _release(eng, insts, slots)
