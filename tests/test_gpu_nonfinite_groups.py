"""NaN and infinite particles in the passes that give a particle a group of lanes."""
import numpy as np
import pytest

from sph_amd import BatchedSPH, NaiveSPHStrategy, VoxelSPHStrategy
from sph_amd.data_classes import SimulationState
from sph_amd.workloads import box_uniform, voxel_for

pytestmark = pytest.mark.gpu

TOL = 1e-5  # of a density, as for the other lane counts


def spoilt(pos, vel, seed):
    """Every seventeenth particle with a NaN or infinite coordinate or velocity component."""
    rng = np.random.default_rng(seed)
    pos, vel = pos.copy(), vel.copy()
    for i in range(0, len(pos), 17):
        a = (pos, pos, vel)[i % 3]
        a[i, rng.integers(3)] = (np.nan, np.inf, -np.inf)[rng.integers(3)]
    return pos, vel


# 16 and 8 lanes that sum in one lane's order; 30 neighbours, past the list's slots and past its tail
@pytest.mark.parametrize("n,mean", [(35, 30), (3001, 30), (3001, 150), (3001, 400), (30011, 130)])
def test_ordered_groups(gpu, n, mean):
    h = min(0.1, (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0))
    w = box_uniform(n, seed=131, h=h)
    pos, vel = spoilt(w.state.position, np.random.default_rng(132).normal(0.0, 0.3, size=(n, 3)), 133)
    state = SimulationState(pos, vel, np.zeros(n))
    batch = BatchedSPH([(w.params, w.constants)], device=gpu)  # one lane per particle
    batch.upload([state])
    batch.step(2)
    want = batch.download()[0]
    got = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu, check_finite=False).advance(state, 2)
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(want, f), equal_nan=True), f


# the four particles of a wavefront search together where all have more than 192 neighbours
@pytest.mark.parametrize("n,mean,scale", [(1603, 500, 1.0), (2999, 700, 0.5)])
def test_shared_rows(gpu, n, mean, scale):
    h = min(0.3, (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0))
    w = box_uniform(n, seed=134, h=h)
    pos, vel = spoilt(w.state.position, np.random.default_rng(135).normal(0.0, 0.3, size=(n, 3)), 136)
    state = SimulationState(pos, vel, np.zeros(n))
    one, got = [NaiveSPHStrategy(w.params, constants=w.constants, device=gpu, grid_voxel=voxel_for(h) * scale, lanes=lanes,
                                 check_finite=False).compute_next_state(state) for lanes in (1, 16)]
    assert np.max(np.abs(got.density - one.density) / np.maximum(one.density, 1.0)) <= TOL
    assert np.array_equal(got.density == 0.0, ~np.isfinite(pos).all(1))
    for f in ("position", "velocity"):
        assert np.array_equal(np.isfinite(getattr(got, f)), np.isfinite(getattr(one, f))), f


# 32 lanes per particle of the VOXEL formulation against one, which particles far away bring about
@pytest.mark.parametrize("n,mean", [(35, 30), (3001, 30), (3001, 60)])
def test_voxel_groups(gpu, n, mean):
    most = 98305
    h = min(0.05, (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0))
    w = box_uniform(most, seed=137, h=h)
    rng = np.random.default_rng(138)
    pos, vel = w.state.position, rng.normal(0.0, 0.3, size=(most, 3))
    pos[n:] = rng.uniform(0.6, 0.95, size=(most - n, 3))
    pos[:n], vel[:n] = spoilt(pos[:n], vel[:n], 139)
    one, got = [VoxelSPHStrategy(box_uniform(count, h=h).params, constants=w.constants, device=gpu, check_finite=False).advance(
        SimulationState(pos[:count], vel[:count], np.zeros(count)), 1) for count in (most, n)]
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(one, f)[:n], equal_nan=True), f
