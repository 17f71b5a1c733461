"""The capped hydrogen-bond count of points without the chessboard, taken on
the device.  Bar: whole numbers equal to the sequential count (the reference's
loop over cells in index order)."""
import numpy as np
import pytest

from cvfbulkwater_amd import FP32_COMPENSATED, VOLUME_DEVICE, Params, Simulation

pytestmark = pytest.mark.gpu


def sequential_count(L, sigma):
    """2 N_HB, at most four bonds per cell (gpu_water3D.cu:2064-2099)."""
    s = sigma.reshape(6, L, L, L)  # [arm][z][y][x]
    match = np.stack([s[0] == np.roll(s[1], -1, 2), s[2] == np.roll(s[3], -1, 1), s[4] == np.roll(s[5], -1, 0)], -1)
    match = match.reshape(-1, 3).tolist()
    count, n = [0] * L**3, 0
    for c in range(L**3):
        x, y, z = c % L, c // L % L, c // (L * L)
        for a, j in enumerate(((x + 1) % L + L * (y + L * z), x + L * ((y + 1) % L + L * z),
                               x + L * (y + L * ((z + 1) % L)))):
            if match[c][a] and count[c] < 4 and count[j] < 4:
                count[c] += 1
                count[j] += 1
                n += 2
    return n


# the smallest workgroup (4), a round of less, exactly and more than one trip
# of 1024 threads (44 / 48), the last size in LDS and the first beyond (52, 56),
# points of both rules and several sizes
@pytest.mark.parametrize("Ls,rules", [([4], [0]), ([8], [0]), ([12], [0]), ([44], [0]), ([48], [0]), ([52], [0]),
                                      ([56], [0]), ([8, 4, 12, 8], [0, 1, 0, 0]), ([60, 8], [0, 0])])
def test_capped_count_equals_sequential(Ls, rules):
    sim = Simulation([Params(L=L, T=0.7, P=0.3, seed=23 + i, flag_chessboard=r, precision=FP32_COMPENSATED,
                             volume_mode=VOLUME_DEVICE) for i, (L, r) in enumerate(zip(Ls, rules))])
    rng = np.random.default_rng(7)
    # random arms (few bonds), one value everywhere (every bond matches), mostly one value, after steps
    for fill in ("random", "one", "most", "steps"):
        if fill == "steps":
            sim.step(3)
        for i, (L, r) in enumerate(zip(Ls, rules)):
            if r:
                continue
            if fill != "steps":
                n = 6 * L**3
                s = {"random": rng.integers(0, 6, n), "one": np.full(n, 3),
                     "most": np.where(rng.random(n) < 0.85, 2, rng.integers(0, 6, n))}[fill].astype(np.uint8)
                sim.set_config(s, sim.get_config(i)[1], i)
        for i, (L, r) in enumerate(zip(Ls, rules)):
            if not r:
                assert sim.observe(i).nhb2 == sequential_count(L, sim.get_config(i)[0]), (fill, i)
