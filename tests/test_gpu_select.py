"""Merges with many improving rows, whose greedy subset is selected without a
sort of all of them (csrc/mlp_kernels.hip select_spans, select_swaps), against
the oracle's serial greedy: the kept moves in their order, the tour, the
latency.

Sizes around the workgroups' threads and the LDS buffer's capacities, both row
maps, LDS and device-memory working arrays; a tour whose swaps conflict in one
chain in the order of their costs, and one with hundreds of spans of nearly
equal cost (the selections then leave the merge to the whole sort).  Whole
numbers: no tolerance.
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


def _check(eng, xs, ys, tour, rowmap, force=False, nbs=range(5)):
    inst = eng.instance(xs, ys, 1)
    s = eng.slot(inst)
    eng.merge_force_global(force)
    try:
        for nb in nbs:
            ref = O.eval_rows_xy(nb, rowmap, xs, ys, 1, tour)
            imp = np.flatnonzero(ref["cost"] < 0)
            kept, _ = O.merge(nb, ref["cost"], ref["i"], ref["j"])
            want = [(int(ref["cost"][r]), nb, int(ref["i"][r]), int(ref["j"][r]), int(r)) for r in kept]
            t2 = tour.copy()
            for _, _, i, j, _ in want:
                t2 = O.apply(nb, t2, i, j)
            eng.set_tour(s, tour)
            eng.eval([s], 1 << nb, rowmap)
            eng.merge_apply([s], nb)
            got = eng.applied(s, nb)
            assert [m[0] for m in got] == [m[0] for m in want], (nb, len(imp))
            assert got == want, (nb, len(imp))
            assert np.array_equal(eng.get_tour(s), t2), (nb, len(imp))
            assert int(eng.latency([s])[0]) == O.latency_xy(xs, ys, 1, t2), nb
    finally:
        eng.merge_force_global(False)
        eng.destroy_slot(s)
        eng.destroy_instance(inst)


@pytest.mark.parametrize("rowmap", [0, 1])
@pytest.mark.parametrize("n", [70, 255, 256, 257, 258, 300, 511, 512, 513, 1022, 1023, 1024, 1025, 1026,
                               2046, 2047, 2049, 3001, 4095, 4097, 5600, 6400])
def test_random_tours(eng, n, rowmap):
    xs, ys = (O.instance_clustered if n % 2 else O.instance_uniform)(n, 70 + n)
    _check(eng, xs, ys, O.perm_tour(n, n), rowmap)


@pytest.mark.parametrize("rowmap", [0, 1])
@pytest.mark.parametrize("n", [60, 130, 270, 1000, 9001, 10500])
def test_device_memory_arrays(eng, n, rowmap):
    xs, ys = O.instance_clustered(n, 90 + n)
    _check(eng, xs, ys, O.perm_tour(n, n), rowmap, force=True, nbs=range(5) if n < 2000 else (0, 1, 3))


@pytest.mark.parametrize("force", [False, True])
@pytest.mark.parametrize("n", [120, 200, 300, 600, 1500])
def test_chain_of_swaps(eng, n, force):
    """A line with every third client off it, by an amount that grows with the
    position: each swap conflicts with the next, their costs in order (53
    rounds of the selection at n = 600)."""
    p = np.arange(n)
    _check(eng, (20 * p).astype(np.int32), np.where(p % 3 == 1, 5 + p, 0).astype(np.int32),
           np.concatenate([p, [0]]).astype(np.int32), 0, force)


@pytest.mark.parametrize("force", [False, True])
@pytest.mark.parametrize("n,w", [(3001, 2), (3001, 4), (6001, 3), (6001, 8)])
def test_nearly_equal_costs(eng, n, w, force):
    """A line in windows of w rotated by one: from the second slice on one
    class of costs holds thousands of spans."""
    p = np.arange(n)
    perm = np.concatenate([[0]] + [np.roll(np.arange(q, min(q + w, n)), 1) for q in range(1, n, w)])
    _check(eng, (3 * p).astype(np.int32), (0 * p).astype(np.int32),
           np.concatenate([perm, [0]]).astype(np.int32), 0, force)
