"""One-plane resident slabs of the reference schedule (the kernel that lays the
moves of a batch of half-sweeps out ahead).  Bar: lattices and volumes bit-exact
against the same steps on the unfused kernels, which the parity tests hold to
the oracle."""
import numpy as np
import pytest

from cvfbulkwater_amd import FP32_COMPENSATED, VOLUME_DEVICE, Params, Simulation

pytestmark = pytest.mark.gpu


# fewer cells than one wave (4), records of all twelve half-sweeps (12 at 256
# threads), of six (56), four (32 at 256) and two (20 at 64), one trip and several
# of the lanes, two workgroups per CU, the last lattice of the kernel and the
# first of the general one (56, 60), a cluster sweep
@pytest.mark.parametrize("Ls,nc,streams,block", [
    ([4], 0, 1, 64), ([4], 0, 1, 1024), ([12], 0, 1, 256), ([20], 0, 1, 64), ([20], 0, 1, 256), ([24], 0, 1, 512),
    ([32], 0, 1, 512), ([32], 0, 1, 256), ([44], 0, 1, 1024), ([56], 0, 1, 1024), ([60], 0, 1, 1024),
    ([16, 28], 0, 2, 256), ([8, 4, 12, 8], 0, 1, 128), ([12, 16], 1, 1, 256)])
def test_planes_equal_unfused(Ls, nc, streams, block):
    pts = [Params(L=L, T=0.6 + 0.03 * i, P=0.3, seed=71 + i, n_cluster=nc, precision=FP32_COMPENSATED,
                  volume_mode=VOLUME_DEVICE) for i, L in enumerate(Ls)]
    a, b = Simulation(pts), Simulation(pts)
    a.tuning = {"fused": 2, "streams": streams, "slab_planes": 1, "block_chunk": block, "graph_steps": 64}
    b.tuning = {"fused": 0, "streams": 1}
    assert a.plan(0)["kind"] == "resident" and a.plan(0)["slab_planes"] == 1
    # calls that begin at every place of the four steps' schedule, and longer ones
    for n in (1, 2, 3, 4, 5, 13, 70):
        a.step(n)
        b.step(n)
        for i in range(len(Ls)):
            x, y = a.get_config(i), b.get_config(i)
            assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), (n, i)
            assert a.volume(i) == b.volume(i)


# as many half-sweeps' records at a time as a workgroup's share of LDS holds: four
# (16 at 64 threads), three (36 at 256, 52 at 512), two (28 at 128, 40 at 256), one
# (32 at 128, 44 and 48 at 256)
@pytest.mark.parametrize("L,block", [(16, 64), (36, 256), (52, 512), (28, 128), (40, 256), (32, 128), (44, 256),
                                     (48, 256)])
def test_few_records_at_a_time(L, block):
    p = Params(L=L, T=0.7, P=0.3, seed=91, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE)
    a, b = Simulation(p), Simulation(p)
    a.tuning = {"fused": 2, "streams": 1, "slab_planes": 1, "block_chunk": block, "graph_steps": 64}
    b.tuning = {"fused": 0, "streams": 1}
    assert a.plan(0)["kind"] == "resident" and a.plan(0)["slab_planes"] == 1
    for n in (1, 6, 70):
        a.step(n)
        b.step(n)
        x, y = a.get_config(), b.get_config()
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), n
        assert a.volume() == b.volume()
