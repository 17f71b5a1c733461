"""The fast schedule in the resident kernel (two colour passes, one exchange of
boundary planes between them).  Bar: lattices and volumes bit-exact against the
same steps on the per-pass kernels, which test_gpu_fast_schedule.py holds to the
oracle."""
import numpy as np
import pytest

from cvfbulkwater_amd import FP32_COMPENSATED, SCHED_FAST, VOLUME_DEVICE, Params, Simulation

pytestmark = pytest.mark.gpu


# whole-lattice windows (many points, a workgroup of several slabs), one-plane
# slabs (4, 12, 32, 68: fewer and more quads than lanes), slabs of two planes
# and more (streams = 2: two workgroups per CU), a cluster sweep (one step a launch)
@pytest.mark.parametrize("Ls,nc,streams,slab,block", [
    ([4], 0, 1, 1, 64), ([4], 0, 1, 0, 256), ([12], 0, 1, 1, 256), ([32], 0, 1, 1, 512), ([32], 0, 1, 2, 256),
    ([68], 0, 1, 1, 1024), ([16, 24], 0, 2, 0, 512), ([16, 24], 1, 1, 1, 1024), ([48, 4, 12, 48], 0, 1, 4, 1024),
    ([8, 12, 16, 20] * 20, 0, 1, 0, 1024)])
def test_fast_resident_equals_per_pass_kernels(Ls, nc, streams, slab, block):
    pts = [Params(L=L, T=0.55 + 0.005 * i, P=0.3, seed=61 + i, n_cluster=nc, schedule=SCHED_FAST,
                  precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE) for i, L in enumerate(Ls)]
    a, b = Simulation(pts), Simulation(pts)
    a.tuning = {"fused": 2, "streams": streams, "slab_planes": slab, "block_chunk": block, "graph_steps": 8}
    b.tuning = {"fused": 0, "streams": 1}
    assert a.plan(0)["kind"] == "resident" and b.plan(0)["kind"] == "unfused"
    for n in (1, 2, 13):
        a.step(n)
        b.step(n)
        for i in range(len(Ls)):
            x, y = a.get_config(i), b.get_config(i)
            assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), (n, i)
            assert a.volume(i) == b.volume(i)
