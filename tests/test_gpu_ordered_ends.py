"""Groups of lanes that sum in one lane's order, at the ends of the terms that they hand each other."""
import numpy as np
import pytest

from sph_amd import BatchedSPH, NaiveSPHStrategy
from sph_amd.data_classes import SimulationState
from sph_amd.workloads import box_uniform

pytestmark = pytest.mark.gpu

H = 0.02


def clusters(counts, seed):
    """Clusters of the given numbers of particles, all of a cluster within H of each other, at
    random places of the order of ids."""
    rng = np.random.default_rng(seed)
    side = int(np.ceil(len(counts) ** (1.0 / 3.0)))
    pos = []
    for c, k in enumerate(counts):
        centre = 0.1 + 3.0 * H * np.array([c % side, c // side % side, c // side ** 2])
        pos.append(centre + rng.uniform(-0.25 * H, 0.25 * H, size=(k, 3)))
    return rng.permutation(np.concatenate(pos))


# sums of 1 to 20 terms end on every place of a group of four; of 90 to 100 around the list's 96 slots;
# of 118 to 130 around the 124 terms that are kept between two additions, 240 to 250 around twice that.
# Up to 24,576 particles have 16 lanes each, up to 98,304 have 8.
@pytest.mark.parametrize("ranges,copies", [([(1, 21)], 10), ([(1, 21)], 130), ([(90, 101), (118, 131)], 3),
                                           ([(90, 101), (118, 131)], 12), ([(240, 251)], 4), ([(240, 251)], 12)])
def test_ends_of_the_terms(gpu, ranges, copies):
    pos = clusters([k for a, b in ranges for k in range(a, b)] * copies, 95)
    n = len(pos)
    w = box_uniform(n, seed=96, h=H)
    state = SimulationState(pos, np.random.default_rng(97).normal(0.0, 0.01, size=(n, 3)), np.zeros(n))
    batch = BatchedSPH([(w.params, w.constants)], device=gpu)  # one lane per particle
    batch.upload([state])
    batch.step(1)
    want = batch.download()[0]
    got = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu).advance(state, 1)
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(want, f)), f
