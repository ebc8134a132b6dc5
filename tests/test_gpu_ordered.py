"""Groups of lanes that sum in one lane's order: the same bits as the one-lane kernels."""
import numpy as np
import pytest

from sph_amd import BatchedSPH, NaiveSPHStrategy
from sph_amd.data_classes import SimulationState
from sph_amd.workloads import box_uniform

pytestmark = pytest.mark.gpu


# a batch of one instance runs the one-lane kernels whatever its size; 24,576 and 98,304 are the
# last sizes with 16 and with 8 lanes; 105, 150 and 250 neighbours are past the 96 list slots (150
# and 250 also past the 124 terms kept between two additions)
@pytest.mark.parametrize("n,mean", [(1, 30), (15, 30), (17, 2), (4096, 30), (3001, 105), (3001, 150), (3001, 250),
                                    (24576, 30), (24577, 30), (30011, 130), (98304, 30), (98305, 30)])
def test_ordered_groups_sum_as_one_lane(gpu, n, mean):
    h = min(0.1, (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0))
    w = box_uniform(n, seed=81, h=h)
    vel = np.random.default_rng(82).normal(0.0, 0.3, size=(n, 3))
    state = SimulationState(w.state.position, vel, np.zeros(n))
    batch = BatchedSPH([(w.params, w.constants)], device=gpu)
    batch.upload([state])
    batch.step(3)
    want = batch.download()[0]
    got = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu).advance(state, 3)
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(want, f)), f


# up to 307,200 particles one lane takes its candidates in threes, past that in pairs, in a batch
# in pairs; 60 neighbours fill the staged list slots, 130 all of them
@pytest.mark.parametrize("n,mean", [(98305, 60), (110003, 130), (307200, 30), (307201, 30)])
def test_threes_and_pairs_sum_alike(gpu, n, mean):
    test_ordered_groups_sum_as_one_lane(gpu, n, mean)
