"""32 lanes per particle take the rows of candidates end to end, and a batch whose instances use
at most 16 lanes has kernels without that path."""
import numpy as np
import pytest

from sph_amd import BatchedSPH, NaiveSPHStrategy
from sph_amd.data_classes import SimulationState
from sph_amd.workloads import box_uniform, voxel_for

pytestmark = pytest.mark.gpu


# scale 1 has 9 rows or fewer around a particle, 0.5 has 25, 0.25 has 81 (three passes of 32); 1 and 31
# particles leave most rows empty, 2,600 neighbours fill several windows from one row
@pytest.mark.parametrize("lanes", [16, 32])
@pytest.mark.parametrize("n,mean,scale", [(1, 30, 1.0), (31, 4, 0.5), (33, 40, 0.25), (3001, 12, 0.5), (3001, 30, 1.0),
                                          (3001, 110, 0.25), (3001, 250, 0.5), (6007, 2600, 1.0)])
def test_windows_over_rows_find_every_neighbour(gpu, lanes, n, mean, scale):
    h = min(0.2, (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0))
    w = box_uniform(n, seed=83, h=h)
    state = SimulationState(w.state.position, np.random.default_rng(84).normal(0.0, 0.3, size=(n, 3)), np.zeros(n))

    def plain(count, steps):
        sim = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu, grid_voxel=voxel_for(h) * scale, lanes=count)
        return sim.advance(state, steps)

    # a density is a sum of up to n positive terms: two orders of it differ by 2 (n - 1) roundings
    # of 2^-24 at most, plus one each of the factor and the result
    want, got = plain(1, 1), plain(lanes, 1)
    assert np.all(np.abs(got.density - want.density) <= 2.0 * (n + 2) * 2.0 ** -24 * want.density)
    batch = BatchedSPH([(w.params, w.constants)], device=gpu, cell_scale=[scale], lanes=[lanes])
    batch.upload([state])
    batch.step(3)
    got, want = batch.download()[0], plain(lanes, 3)
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(want, f)), f


# groups of 2 and 4 lanes look a batch ahead up to 270,000 threads and in batches: the same bits
@pytest.mark.parametrize("lanes,n", [(2, 135000), (2, 135001), (4, 67500), (4, 67501)])
def test_plain_groups_and_batches_sum_alike(gpu, lanes, n):
    h = (30 / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0)
    w = box_uniform(n, seed=87, h=h)
    state = SimulationState(w.state.position, np.random.default_rng(88).normal(0.0, 0.3, size=(n, 3)), np.zeros(n))
    batch = BatchedSPH([(w.params, w.constants)], device=gpu, lanes=[lanes])
    batch.upload([state])
    batch.step(2)
    got = batch.download()[0]
    want = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu, lanes=lanes).advance(state, 2)
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(want, f)), f
