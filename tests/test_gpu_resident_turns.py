"""Resident launches of several handles whose plans do not fit on the card
together."""
import threading
import time

import pytest

from cvfbulkwater_amd import FP64, SCHED_FAST, VOLUME_HOST, Params, Simulation

pytestmark = pytest.mark.gpu


def test_a_long_call_lets_another_handle_in():
    """A handle's call of many launches, with the host's volume moves between
    them, holds its turn for one launch and not for the call."""
    sims = [Simulation([Params(L=L, T=0.7, P=0.3, seed=5 + i, precision=FP64, volume_mode=VOLUME_HOST)
                        for i, L in enumerate([16] * 65)]) for _ in range(2)]
    for s in sims:
        assert s.plan(0)["kind"] == "resident"
        s.step(1)
        s.sync()
    a, b = sims
    t = threading.Thread(target=a.step, args=(64 * 1500,))
    t.start()
    time.sleep(0.02)
    b.step(1)
    running = t.is_alive()
    t.join()
    assert running
    assert (a.steps, b.steps) == (1 + 64 * 1500, 2)
    for s in sims:
        s.sync()


def test_handles_of_every_kind_side_by_side():
    """Plain and cluster handles, one-plane and whole-card plans, both schedules and
    handles without a resident plan, each sampled by a thread of its own:
    what each gives alone, without a launch that had to be given up."""
    sets = [([32] * 8, dict(n_cluster=1)), ([20] * 24, dict(n_cluster=1)), ([48] * 5, {}),
            ([16, 24, 32, 48] * 8, dict(schedule=SCHED_FAST)), ([12], {}), ([32], dict(flag_chessboard=0))]

    def handle(j):
        Ls, kw = sets[j]
        return Simulation([Params(L=L, T=0.7, P=0.3, seed=100 * j + i, precision=FP64, volume_mode=VOLUME_HOST, **kw)
                           for i, L in enumerate(Ls)])

    def sample(s):
        out = []
        for k in range(6):
            s.step(3 + k)
            out.append((s.observe(), s.step_histograms(2).tolist(), s.cluster_stats()))
        return out

    want, got = [], [None] * len(sets)
    for j in range(len(sets)):
        with handle(j) as s:
            want.append(sample(s))
    sims = [handle(j) for j in range(len(sets))]
    kinds = [s.plan()["kind"] for s in sims]

    def run(j):
        got[j] = sample(sims[j])

    threads = [threading.Thread(target=run, args=(j,)) for j in range(len(sets))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got == want
    assert [s.plan()["kind"] for s in sims] == kinds
