"""A sampling interval: any number of steps per call as resident launches,
and one sample kernel per handle (observables, volume states).  Bars: the
observables' integers equal a recount of the lattice, lattices bit-exact
against the same steps taken one by one on the unfused kernels."""
import numpy as np
import pytest

from cvfbulkwater_amd import FP32_COMPENSATED, VOLUME_DEVICE, Params, Simulation

pytestmark = pytest.mark.gpu


def recount(L, sigma, eta):
    """2 N_HB and N_sigma of a lattice (gpu_water3D.cu:2014-2103)."""
    s = sigma.reshape(6, L, L, L).astype(np.int64)  # [arm][z][y][x]
    e = eta.reshape(6, L, L, L).astype(np.int64)
    nhb2 = 0
    for a, ax in ((0, 2), (2, 1), (4, 0)):
        facing_s, facing_e = np.roll(s[a + 1], -1, ax), np.roll(e[a + 1], -1, ax)
        nhb2 += int(((s[a] == facing_s) * (e[a] + facing_e)).sum())
    nsig = sum(int((s[i] == s[j]).sum()) for i in range(6) for j in range(i + 1, 6))
    return nhb2, nsig


# one cell group per thread and workgroup (L = 4: 64 cells), partial and whole
# workgroups, both workgroup spans (2^20 cells between 100 and 104), a mix
@pytest.mark.parametrize("Ls", [[4], [8], [12], [20], [36], [100], [104], [4, 48, 12, 28, 4, 96]])
def test_sample_equals_recount(Ls):
    pts = [Params(L=L, T=0.6 + 0.05 * i, P=0.2, seed=77 + i, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE)
           for i, L in enumerate(Ls)]
    sim = Simulation(pts)
    for steps in (0, 3):
        if steps:
            sim.step(steps)
        for i, L in enumerate(Ls):
            o = sim.observe(i)
            assert (o.nhb2, o.n_sigma) == recount(L, *sim.get_config(i)), (Ls, i, steps)
            assert (o.r_cell, o.E_vdw) == (sim.volume(i)[0], sim.volume(i)[2])
            assert o.step == steps


def test_sample_follows_set_config_and_set_shells():
    sim = Simulation([Params(L=8, seed=5, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE) for _ in range(2)])
    before = sim.observe(1)
    s, e = sim.get_config(1)
    sim.set_config((s + 1) % 6 * (np.arange(s.size) % 2 == 0), e, 1)
    o = sim.observe(1)
    assert (o.nhb2, o.n_sigma) == recount(8, *sim.get_config(1)) and o.n_sigma != before.n_sigma
    d, f = sim.shells(1)
    sim.set_shells(d[:1], f[:1], 1)
    assert sim.observe(1).E_vdw == sim.volume(1)[2] != o.E_vdw


@pytest.mark.parametrize("Ls,graph_steps", [([12], 64), ([16, 24], 64), ([32], 4)])
def test_calls_of_any_length_equal_single_steps(Ls, graph_steps):
    """10 = 8 + 2, 65 = 64 + 1 and longer calls as single resident launches
    (at most graph_steps steps each) against the unfused kernels."""
    pts = [Params(L=L, T=0.7, P=0.3, seed=9 + i, precision=FP32_COMPENSATED, volume_mode=VOLUME_DEVICE)
           for i, L in enumerate(Ls)]
    a, b = Simulation(pts), Simulation(pts)
    a.tuning = {"fused": 2, "slab_planes": 1, "graph_steps": graph_steps}
    b.tuning = {"fused": 0}
    for n in (1, 10, 65, 3, 130):
        a.step(n)
        b.step(n)
        for i in range(len(Ls)):
            x, y = a.observe(i), b.observe(i)
            assert x == y, (n, i)
            assert all(np.array_equal(u, v) for u, v in zip(a.get_config(i), b.get_config(i))), (n, i)
    # the step counter serves the other plans after the resident launches
    a.tuning = {"fused": 1, "slab_planes": 0}
    a.step(5)
    b.step(5)
    assert all(a.observe(i) == b.observe(i) for i in range(len(Ls)))
