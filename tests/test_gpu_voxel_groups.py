"""VOXEL density and force by 32 lanes per particle, which few particles take, against the one-lane
kernels."""
from dataclasses import replace

import numpy as np
import pytest

from sph_amd.data_classes import SimulationState
from sph_amd.strategy import VoxelSPHStrategy
from sph_amd.workloads import box_uniform

pytestmark = pytest.mark.gpu

ONE_LANE = 98305  # the fewest particles of the one-lane density kernel; the force kernel's are 32,769


# 2 and 60 neighbours end before and after the 32 a list holds; "pile" puts all particles into one
# voxel, "outside" some out of the grid, whose keys wrap (no voxel may be skipped then)
@pytest.mark.parametrize("n,mean,form", [(1, 30, ""), (7, 2, ""), (9, 60, ""), (3001, 2, ""), (3001, 30, ""), (3001, 60, ""),
                                         (700, 30, "pile"), (3001, 30, "outside"), (32768, 60, ""), (32769, 30, ""),
                                         (98303, 30, "")])
@pytest.mark.parametrize("block", [64, 256])
def test_voxel_groups_equal_one_lane(gpu, n, mean, form, block):
    """Particles too far away to be anyone's neighbour bring the state past the group kernel's range;
    the others' lists keep their order, so the step's bits are the same (a particle that lists only
    itself has a density of zero and no finite step)."""
    h = min(0.05, (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0))
    w = box_uniform(ONE_LANE, seed=85, h=h)
    rng = np.random.default_rng(86)
    pos, vel = w.state.position, rng.normal(0.0, 0.3, size=(ONE_LANE, 3))
    pos[n:] = rng.uniform(0.6, 0.95, size=(ONE_LANE - n, 3))
    if form == "pile":
        pos[:n] = h * rng.uniform(8.05, 8.95, size=(n, 3))
    if form == "outside":
        pos[:n:7, 0] = rng.uniform(-0.08, 0.0, size=len(pos[:n:7]))
        pos[3:n:50, 1] = rng.uniform(1.0, 1.05, size=len(pos[3:n:50]))

    def run(count):
        params = box_uniform(count, h=h).params
        sim = VoxelSPHStrategy(params, constants=w.constants, device=gpu, launch=(block, 256), check_finite=False)
        return sim.advance(SimulationState(pos[:count], vel[:count], np.zeros(count)), 1)

    want, got = run(ONE_LANE), run(n)
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(want, f)[:n], equal_nan=True), f


# with h from 0.5 to 0.95 of the voxel's edge up to 131,072 particles have groups, below that 307,200
@pytest.mark.parametrize("n,edges,most", [(131072, 0.7, 131072), (20011, 0.7, 131072), (307200, 0.4, 307200),
                                          (20011, 0.2, 307200)])
def test_coarse_voxels_equal_one_lane(gpu, n, edges, most):
    h = (30 / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0)
    w = box_uniform(most + 1, seed=89, h=h)
    rng = np.random.default_rng(90)
    pos, vel = w.state.position, rng.normal(0.0, 0.3, size=(most + 1, 3))
    pos[n:] = rng.uniform(0.7, 0.95, size=(most + 1 - n, 3))

    def run(count):
        params = replace(box_uniform(count, h=h).params, voxel_size=np.array([h / edges] * 3))
        sim = VoxelSPHStrategy(params, constants=w.constants, device=gpu, check_finite=False)
        return sim.advance(SimulationState(pos[:count], vel[:count], np.zeros(count)), 1)

    want, got = run(most + 1), run(n)
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(want, f)[:n], equal_nan=True), f
