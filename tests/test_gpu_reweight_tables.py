"""Constants' sweeps on tables of exponentials: numbers of simulations around
the kernels' paddings, cells whose targets use different sums (3000 samples:
arguments on both sides of the cut at 10), exponents from near zero to the
largest that the tables serve, and beyond it.  Constants against the oracle to
1e-9 absolute: arguments of up to 10^6 with a rounding of 1e-16 each."""
import numpy as np
import pytest

from cvfbulkwater_amd.reweight import Reweighting
from oracle import rw
import rw_synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_sim,n,span,L,bf", [
    (2, 3000, 0.001, 8, 1.0), (3, 3000, 0.004, 8, 0.5), (7, 3000, 0.001, 8, 0.5), (15, 500, 0.002, 8, 0.5),
    (16, 1500, 0.01, 8, 0.5), (16, 1500, 0.0, 8, 0.5),
    # shifts of about 40, 80 and 400 (exponentials in every cell)
    (4, 1000, 0.01, 8, 0.5), (4, 1000, 0.02, 8, 0.5), (4, 1000, 0.1, 8, 0.5), (4, 1000, 0.004, 16, 0.5),
    (2, 9, 0.001, 4, 0.5), (17, 500, 0.001, 8, 0.5)])
def test_constants_match_oracle(n_sim, n, span, L, bf):
    Ts = [0.1058 + span * k / max(n_sim - 1, 1) for k in range(n_sim)]
    Ps = [0.5 + 0.0005 * (k % 3) for k in range(n_sim)]
    data = rw_synth.samples(Ts, n, seed=11 + n_sim)
    ora = rw.OraGrid.from_samples(L, Ts, Ps, [n] * n_sim, np.concatenate(data), bf)
    with Reweighting(L, Ts, Ps, data, bf) as eng:
        for steps in (1, 3, 12):
            c, prev, ok = eng.solve_constants(steps)
            co, po, rc = ora.constants(steps)
            np.testing.assert_allclose(c, co, rtol=0, atol=1e-9)
            np.testing.assert_allclose(prev, po, rtol=0, atol=1e-9)
            assert ok == (rc == 0)
            again = eng.solve_constants(steps)
            assert np.array_equal(again[0], c) and np.array_equal(again[1], prev)
    ora.close()
