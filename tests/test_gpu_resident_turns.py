"""Resident launches of several handles whose plans do not fit on the card
together."""
import threading
import time

import pytest

from cvfbulkwater_amd import FP64, VOLUME_HOST, Params, Simulation

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
