"""A server's jobs when the context's round form changes between its steps:
the form of a round is a setting of the context, which the program may change
at any time, and every job's result stays the oracle's DVND result.

The rounds that leave out blocks of moves (csrc/mlp_prune.h) read summaries of
the tour's blocks, so the rounds of every other form have to keep them up to
date.  Whole numbers: no tolerance.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

wm = pytest.importorskip("wamca_mi")
from wamca_mi import serve  # noqa: E402


@pytest.fixture(scope="module")
def eng():
    e = wm.Engine(0)
    yield e
    e.close()


FORMS = {
    "fused": (lambda e: e.dvnd_fused(True), lambda e: e.dvnd_fused(False)),
    "persistent": (lambda e: e.dvnd_config(4, True, True), lambda e: e.dvnd_config()),
    "tile": (lambda e: e.set_tile(1), lambda e: e.set_tile(-1)),
    "device_memory_merges": (lambda e: e.merge_force_global(True), lambda e: e.merge_force_global(False)),
}


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("sizes", [(300,), (257, 400, 90)])
def test_form_changed_between_steps(eng, form, sizes):
    on, off = FORMS[form]
    jobs, refs = [], []
    for q, n in enumerate(sizes):
        xs, ys = O.instance_uniform(n, 600 + n)
        W = O.weights(xs, ys, 1)
        jobs.append((xs, ys, O.random_tour(O.MT(n), W, 0.5)))
        refs.append(O.dvnd(W, jobs[q][2], 0))
    srv = serve.Server(eng, rounds_per_step=1)
    got, step = {}, 0
    try:
        for q, (xs, ys, t) in enumerate(jobs):
            srv.submit(xs, ys, t, 1, tag=q)
        while len(got) < len(jobs):
            # three steps of the other form, three of the usual one
            (on if step % 6 < 3 else off)(eng)
            srv.step()
            got.update({r["tag"]: r for r in srv.poll()})
            step += 1
    finally:
        off(eng)
        srv.close()
    for q, (tref, Lref, rref, _) in enumerate(refs):
        assert (got[q]["latency"], got[q]["rounds"]) == (Lref, rref), (sizes[q], step)
        assert np.array_equal(got[q]["tour"], tref), sizes[q]
