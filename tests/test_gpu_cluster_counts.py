"""Cluster statistics from the labels.  Bar: whole numbers equal to a count of
the labels on the host, mean and variance as the reference's float sums."""
import numpy as np
import pytest

from cvfbulkwater_amd import FP32_COMPENSATED, VOLUME_DEVICE, Params, Simulation

pytestmark = pytest.mark.gpu


# 6N nodes below, at and above one workgroup's 4096 (4: 384; 8: 3072; 12: 10368),
# several workgroups with a short last one; few bonds, and a lattice whose arms
# all agree, where one cluster holds most nodes and percolates
@pytest.mark.parametrize("L", [4, 8, 12, 20, 44])
@pytest.mark.parametrize("ordered", [False, True])
def test_counts_equal_labels(L, ordered):
    sim = Simulation(Params(L=L, T=0.4 if ordered else 0.8, P=0.2, seed=5 + L, n_cluster=1,
                            precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE))
    for steps in (1, 3):
        if ordered:
            sim.set_config(np.full(6 * L**3, 2, np.uint8), sim.get_config()[1])
        sim.step(steps)
        lab = np.asarray(sim.labels()).ravel()
        roots, size = np.unique(lab, return_counts=True)
        assert np.array_equal(lab[roots], roots)
        c = sim.cluster_stats()
        top = np.sort(size)[::-1]
        assert (c.n_clusters, c.largest, c.second) == (len(size), top[0], top[1] if len(top) > 1 else 0)
        nodes = np.arange(lab.size) % L**3
        perc = 0
        for r in roots[size >= 2 * L]:
            cell = nodes[lab == r]
            perc += any(len(np.unique(v)) == L for v in (cell % L, cell // L % L, cell // (L * L)))
        assert c.n_perc == perc
        total = squares = np.float32(0)
        for s in size:  # in label order
            total += np.float32(s)
            squares += np.float32(s) * np.float32(s)
        mean = total / np.float32(len(size))
        assert c.mean == mean and c.var == squares / np.float32(len(size)) - mean * mean
