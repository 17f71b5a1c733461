"""Default plans by handle size, and resident launches of several handles at
once.  Bar: lattices bit-exact against the unfused kernels."""
import threading

import numpy as np
import pytest

from cvfbulkwater_amd import FP32_COMPENSATED, VOLUME_DEVICE, Params, Simulation

pytestmark = pytest.mark.gpu


def handle(Ls, seed, **kw):
    return Simulation([Params(L=L, T=0.6 + 0.01 * (i % 20), P=0.3, seed=seed + i, precision=FP32_COMPENSATED,
                              volume_mode=VOLUME_DEVICE, **kw) for i, L in enumerate(Ls)])


# 256 planes and one more (one, two workgroups per CU), three, four, more planes
# than that (thicker slabs), lattices too small for those, a cluster sweep
@pytest.mark.parametrize("Ls,nc,streams,slab,kind", [
    ([32] * 8, 0, 1, 1, "resident"), ([32] * 8 + [4], 0, 2, 1, "resident"), ([24] * 24, 0, 3, 1, "resident"),
    ([16] * 60, 0, 4, 1, "resident"), ([16] * 65, 0, 1, 0, "resident"), ([8] * 130, 0, 1, 0, "fused"),
    ([48] * 6, 0, 1, 0, "resident"), ([20] * 20, 1, 2, 1, "resident"), ([48], 1, 1, 0, "fused")])
def test_default_plan(Ls, nc, streams, slab, kind):
    a, b = handle(Ls, 5, n_cluster=nc), handle(Ls, 5, n_cluster=nc)
    assert a.plan(0)["kind"] == kind
    assert (a.tuning["streams"], a.tuning["slab_planes"]) == (streams, slab)
    b.tuning = {"fused": 0, "streams": 1}
    for n in (1, 6):
        a.step(n)
        b.step(n)
    for i in range(0, len(Ls), 7):
        x, y = a.get_config(i), b.get_config(i)
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), i
        assert a.volume(i) == b.volume(i)


def test_resident_handles_of_several_threads():
    """Handles that do not fit on the card together, each stepped by a thread
    of its own, as often as the others allow."""
    sets = [[32] * 16, [48] * 5, [16] * 40, [12], [16, 24, 32, 48] * 8]
    want = []
    for j, Ls in enumerate(sets):
        s = handle(Ls, 100 * j)
        s.step(40)
        want.append([s.get_config(i) for i in range(len(Ls))])
        s.close()
    sims = [handle(Ls, 100 * j) for j, Ls in enumerate(sets)]
    failed = []

    def run(s):
        try:
            for _ in range(10):
                s.step(4)
            s.sync()
        except Exception as e:  # noqa: BLE001 - reported below
            failed.append(repr(e))

    threads = [threading.Thread(target=run, args=(s,)) for s in sims]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    for s, w in zip(sims, want):
        for i, (sigma, eta) in enumerate(w):
            x = s.get_config(i)
            assert np.array_equal(x[0], sigma) and np.array_equal(x[1], eta), i
