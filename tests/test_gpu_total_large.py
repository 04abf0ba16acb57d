"""TOTAL merges of long tours on both sides of the size up to which the merge's
tours stay in LDS (about 5900 positions beside the merge's 104 KB of shared
arrays), against the oracle: the kept moves in their order, the applied tour and
its latency.  Whole numbers: no tolerance."""
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


@pytest.mark.parametrize("n", [5600, 5900, 6100, 7001])
def test_merge_total(eng, n):
    xs, ys = O.instance_uniform(n, n)
    W = O.weights(xs, ys, 1)
    inst = eng.instance(xs, ys, 1)
    s = eng.slot(inst)
    try:
        for nb, block in ((0, 3), (1, 64), (3, 5)):
            t = O.perm_tour(nb + 1, n)
            eng.set_tour(s, t)
            eng.eval_total([s], nb, block)
            ref = O.eval_total(nb, W, t, block)
            kept, _ = O.merge(nb, ref["cost"], ref["i"], ref["j"])
            eng.merge_total([s])
            got = eng.applied(s, nb)
            assert [g[4] for g in got] == kept.tolist(), nb
            assert [(g[0], g[2], g[3]) for g in got] == [
                (int(ref["cost"][q]), int(ref["i"][q]), int(ref["j"][q])) for q in kept], nb
            for q in kept:
                t = O.apply(nb, t, int(ref["i"][q]), int(ref["j"][q]))
            assert np.array_equal(eng.get_tour(s), t), nb
            assert int(eng.latency([s])[0]) == O.latency_xy(xs, ys, 1, t), nb
    finally:
        eng.destroy_slot(s)
        eng.destroy_instance(inst)
