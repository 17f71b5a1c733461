"""Configurations in and out on the device: packed words, cube decoding and
the non-chessboard counters against the oracle, the range errors, and a
lattice that stays as it was when its input is refused."""
import numpy as np
import pytest

from cvfbulkwater_amd import CVFError, Params, Simulation
from oracle import py as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chessboard", [1, 0])
@pytest.mark.parametrize("L", [4, 8, 12, 28, 36])
def test_random_input_decodes_as_the_oracle(L, chessboard):
    rng = np.random.default_rng(L)
    n = 6 * L ** 3
    sim = Simulation(Params(L=L, T=0.7, P=0.2, seed=3, flag_chessboard=chessboard))
    ora = O.OracleSim(L=L, T=0.7, P=0.2, seed=3, flag_chessboard=chessboard)
    solved = sim.get_config()[1]  # a solution's eta, then noise on it, then noise alone
    for eta in (solved, solved ^ (rng.random(n) < 0.01), rng.integers(0, 2, n)):
        sigma = rng.integers(0, 6, n).astype(np.uint8)
        bad = sim.set_config(sigma, eta.astype(np.uint8))
        assert bad == ora.set_config(sigma, eta.astype(np.uint8))
        for t in range(3):
            (s, e), (so, eo) = sim.get_config(), ora.get_config()
            assert np.array_equal(s, so) and np.array_equal(e, eo), (L, chessboard, t)
            a, b = sim.observe(), ora.measure()
            assert (a.nhb2, a.n_sigma) == (b.nhb2, b.n_sigma)
            sim.step(1)
            ora.step(1)


def test_out_of_range_values_are_named_and_change_nothing():
    sim = Simulation([Params(L=8, seed=4), Params(L=12, seed=5)])
    sim.step(2)
    before = [sim.get_config(i) for i in range(2)]
    s, e = (v.copy() for v in before[1])
    N = 12 ** 3
    e[5 * N + 17] = 2
    with pytest.raises(CVFError, match=r"active_bond \(2\) appeared in line 17"):
        sim.set_config(s, e, 1)
    s[2 * N + 40], s[3 * N + 1], e[2 * N + 40] = 255, 6, 7
    with pytest.raises(CVFError, match=r"spin \(255\) appeared in line 40"):
        sim.set_config(s, e, 1)
    for i in range(2):
        assert all(np.array_equal(a, b) for a, b in zip(sim.get_config(i), before[i]))
