"""Fused launches on tiles (folded boxes with a halo found from the launch's
schedule).  Bar: lattices and volumes bit-exact against the same steps on the
unfused kernels, which the parity tests hold to the oracle."""
import numpy as np
import pytest

from cvfbulkwater_amd import FP32_COMPENSATED, VOLUME_DEVICE, Params, Simulation

pytestmark = pytest.mark.gpu


# windows longer than the lattice (4, 8), edges that do not divide it (20, 44,
# 68, 100), one tile per CU and several (128), a mix; both launch lengths, every
# workgroup size the kernel takes, odd and even pass counts, a cluster sweep
@pytest.mark.parametrize("Ls,nm,nc,chunk,block", [
    ([4], 1, 0, 6, 256), ([4], 3, 1, 12, 1024), ([8], 1, 0, 12, 256), ([8], 2, 0, 6, 512),
    ([12], 1, 1, 12, 512), ([20], 1, 0, 6, 256), ([20], 3, 0, 12, 512), ([44], 1, 1, 12, 512),
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


@pytest.mark.parametrize("L,kind,tiled", [(64, "resident", False), (68, "fused", True), (252, "fused", True)])
def test_default_plan_of_wide_lattices(L, kind, tiled):
    plan = Simulation(Params(L=L, seed=3, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE)).plan(0)
    assert plan["kind"] == kind and (plan["slab_planes"] == 0) == tiled


def test_a_requested_slab_thickness_keeps_slabs():
    sim = Simulation(Params(L=32, seed=3, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE))
    sim.tuning = {"fused": 1, "slab_planes": 1}
    assert sim.plan(0)["kind"] == "fused" and sim.plan(0)["slab_planes"] == 1
