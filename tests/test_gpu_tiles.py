"""Fused launches on tiles (folded boxes with a halo found from the launch's
schedule).  Bar: lattices and volumes bit-exact against the same steps on the
unfused kernels, which the parity tests hold to the oracle."""
import numpy as np
import pytest

from cvfbulkwater_amd import FP32_COMPENSATED, VOLUME_DEVICE, Params, Simulation

pytestmark = pytest.mark.gpu


# (a point above L = 64 puts the whole handle on tiles)
# windows longer than the lattice (4, 8), edges that do not divide it (20, 44,
# 68, 100), one tile per CU and several (128), a mix; both launch lengths, every
# workgroup size the kernel takes, odd and even pass counts, a cluster sweep
@pytest.mark.parametrize("Ls,nm,nc,chunk,block", [
    ([4, 68], 1, 0, 6, 256), ([4, 72], 3, 1, 12, 1024), ([8, 68], 1, 0, 12, 256), ([8, 72], 2, 0, 6, 512),
    ([12, 84], 1, 1, 12, 512), ([20, 68], 1, 0, 6, 256), ([20, 76], 3, 0, 12, 512), ([44], 1, 1, 12, 512),
    ([68], 1, 0, 12, 256), ([68], 2, 0, 6, 1024), ([100], 1, 0, 12, 1024), ([128], 1, 0, 6, 512),
    ([4, 68, 12], 1, 0, 6, 256), ([4, 68, 12], 1, 1, 12, 512)])
def test_tiles_equal_unfused(Ls, nm, nc, chunk, block):
    pts = [Params(L=L, T=0.6 + 0.1 * i, P=0.3, seed=41 + i, n_metropolis=nm, n_cluster=nc, precision=FP32_COMPENSATED,
                  volume_mode=VOLUME_DEVICE) for i, L in enumerate(Ls)]
    a, b = Simulation(pts), Simulation(pts)
    a.tuning = {"fused": 1, "slab_planes": 0, "chunk_sweeps": chunk, "block_chunk": block, "streams": 1}
    b.tuning = {"fused": 0}
    for i in range(len(Ls)):
        assert a.plan(i)["kind"] == "fused" and a.plan(i)["slab_planes"] == 0
        assert b.plan(i)["kind"] == "unfused"
    for n in (1, 2, 5):
        a.step(n)
        b.step(n)
        for i in range(len(Ls)):
            x, y = a.get_config(i), b.get_config(i)
            assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), (n, i)
            assert a.volume(i) == b.volume(i)


# without the chessboard a half-sweep's counters need a layer at both ends:
# whole-lattice windows (4, 8), short last tiles (20, 44, 68), both rules at once
@pytest.mark.parametrize("Ls,rules,nm,chunk,block", [
    ([4, 68], [0, 0], 1, 6, 256), ([4, 72], [0, 1], 2, 12, 1024), ([8, 84], [0, 0], 1, 12, 256),
    ([12, 68], [0, 0], 1, 6, 512), ([20, 68], [0, 0], 3, 12, 256), ([32], [0], 1, 6, 512), ([44], [0], 1, 12, 512), ([68], [0], 1, 6, 1024),
    ([68, 8, 12], [0, 1, 0], 1, 12, 256), ([8, 72, 4], [0, 1, 0], 1, 6, 512)])
def test_tiles_without_chessboard_equal_unfused(Ls, rules, nm, chunk, block):
    pts = [Params(L=L, T=0.6 + 0.1 * i, P=0.3, seed=51 + i, n_metropolis=nm, flag_chessboard=r,
                  precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE) for i, (L, r) in enumerate(zip(Ls, rules))]
    a, b = Simulation(pts), Simulation(pts)
    a.tuning = {"fused": 1, "slab_planes": 0, "chunk_sweeps": chunk, "block_chunk": block, "streams": 1}
    b.tuning = {"fused": 0}
    for n in (1, 2, 5):
        a.step(n)
        b.step(n)
        for i in range(len(Ls)):
            assert a.plan(i)["kind"] == "fused" and a.plan(i)["slab_planes"] == 0
            x, y = a.get_config(i), b.get_config(i)
            assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), (n, i)
            assert a.observe(i).nhb2 == b.observe(i).nhb2
            assert a.volume(i) == b.volume(i)


@pytest.mark.parametrize("L,kind,tiled", [(64, "resident", False), (68, "fused", True), (252, "fused", True)])
def test_default_plan_of_wide_lattices(L, kind, tiled):
    plan = Simulation(Params(L=L, seed=3, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE)).plan(0)
    assert plan["kind"] == kind and (plan["slab_planes"] == 0) == tiled


def test_a_requested_slab_thickness_keeps_slabs():
    sim = Simulation(Params(L=32, seed=3, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE))
    sim.tuning = {"fused": 1, "slab_planes": 1}
    assert sim.plan(0)["kind"] == "fused" and sim.plan(0)["slab_planes"] == 1
