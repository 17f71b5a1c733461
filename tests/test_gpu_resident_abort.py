"""Resident launches whose wait for a neighbour timed out, as another process on
the card can bring about: the steps are done again, and no caller sees
it.  Bar: what the unfused kernels give, bit for bit."""
import numpy as np
import pytest

from cvfbulkwater_amd import (FP32_COMPENSATED, FP64, SCHED_FAST, SCHED_REFERENCE, VOLUME_DEVICE, VOLUME_HOST,
                              CVFError, Params, Simulation)

pytestmark = pytest.mark.gpu


def handles(Ls, nc=0, fast=False, device=True):
    pts = [Params(L=L, T=0.6 + 0.03 * (i % 12), P=0.3, seed=171 + i, n_cluster=nc,
                  precision=FP32_COMPENSATED if device else FP64, volume_mode=VOLUME_DEVICE if device else VOLUME_HOST,
                  schedule=SCHED_FAST if fast else SCHED_REFERENCE) for i, L in enumerate(Ls)]
    a, b = Simulation(pts), Simulation(pts)
    b.tuning = {"fused": 0, "streams": 1}
    assert a.plan(0)["kind"] == "resident"
    return a, b


def abort_next(s):
    assert s._lib.cvf_abort_next_launch(s._h) == 0


def same_lattices(a, b):
    for i in range(len(a.params)):
        x, y = a.get_config(i), b.get_config(i)
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]), i
        assert a.volume(i) == b.volume(i)
    assert a.steps == b.steps


# one-plane slabs, thick slabs and whole lattices in one launch (which move on
# where the others give up), the fast schedule, cluster sweeps between the
# launches (which move what the launch left), volume moves on the host
@pytest.mark.parametrize("Ls,nc,fast,device", [
    ([12], 0, False, True), ([32], 0, False, False), ([16, 24, 32, 48] * 8, 0, False, True), ([16] * 65, 0, False, True),
    ([16, 48], 0, True, True), ([8, 20], 1, False, True), ([16], 2, False, False)])
def test_steps_are_done_again(Ls, nc, fast, device):
    a, b = handles(Ls, nc, fast, device)
    plan = a.tuning
    a.step(5)
    abort_next(a)
    a.step(3)  # the aborted launch, and more after it
    a.step(130)
    a.sync()
    assert a.plan(0)["kind"] != "resident"
    b.step(138)
    same_lattices(a, b)
    if nc:
        assert all(np.array_equal(a.labels(i), b.labels(i)) for i in range(len(Ls)))
    # on from there, resident again if asked to, and aborted once more
    a.tuning = plan
    assert a.plan(0)["kind"] == "resident"
    a.step(2)
    abort_next(a)
    a.step(70)
    b.step(72)
    assert [a.observe(i) for i in range(len(Ls))] == [b.observe(i) for i in range(len(Ls))]
    a.step(4)
    b.step(4)
    same_lattices(a, b)


def read_config(a, b):
    same_lattices(a, b)


def read_labels(a, b):
    assert np.array_equal(a.labels(1), b.labels(1))


def load_config(a, b):
    c = b.get_config(0)
    assert a.set_config(c[1] * 0 + 3, c[1], 1) == b.set_config(c[1] * 0 + 3, c[1], 1)


def refuse_config(a, b):
    sigma, eta = b.get_config(1)
    sigma[7] = 6
    for s in (a, b):
        with pytest.raises(CVFError, match="spin"):
            s.set_config(sigma, eta, 1)


def retune(a, b):
    a.tuning = {"fused": 2, "slab_planes": 1, "block_chunk": 128}


def tune(a, b):
    a.autotune(2)


def profile(a, b):
    a.profile_steps(3)
    b.step(3)


def read_clusters(a, b):
    assert a.cluster_stats(1) == b.cluster_stats(1)


def read_histogram(a, b):
    assert np.array_equal(a.sigma_histogram(1), b.sigma_histogram(1))


def record(a, b):
    assert np.array_equal(a.step_histograms(21, 1), b.step_histograms(21, 1))


# the first call after the aborted launch
@pytest.mark.parametrize("call", [read_config, read_labels, load_config, refuse_config, retune, tune, profile,
                                  read_clusters, read_histogram, record], ids=lambda f: f.__name__)
def test_every_call_finds_the_steps_done(call):
    a, b = handles([16, 16], nc=1)
    for s in (a, b):
        s.step(2)
    abort_next(a)
    for s in (a, b):
        s.step(20)
    call(a, b)
    for s in (a, b):
        s.step(2)
    same_lattices(a, b)


# aborted in the first and a later launch of the recorded steps (a launch per step)
@pytest.mark.parametrize("Ls,nc", [([16], 1), ([12, 32], 0)])
@pytest.mark.parametrize("n", [1, 40])
def test_recorded_steps_are_done_again(Ls, nc, n):
    a, b = handles(Ls, nc)
    a.step(3)
    b.step(3)
    abort_next(a)
    assert np.array_equal(a.step_histograms(n, 0), b.step_histograms(n, 0))
    assert np.array_equal(a.step_histograms(5, 0), b.step_histograms(5, 0))
    same_lattices(a, b)
