"""VOXEL density where voxels hold thousands of particles: by 32 lanes per particle only while that
is the faster way, and to the same bits."""
from dataclasses import replace

import numpy as np
import pytest
import torch

from sph_amd.data_classes import SimulationState
from sph_amd.strategy import VoxelSPHStrategy
from sph_amd.workloads import box_uniform

pytestmark = pytest.mark.gpu

MOST = 307200  # no more particles have 32 lanes each, whatever the voxels


def strategy(n, h, edges, gpu):
    w = box_uniform(n, seed=141, h=h)
    params = replace(w.params, voxel_size=np.array([h / edges] * 3))
    return VoxelSPHStrategy(params, constants=w.constants, device=gpu, check_finite=False), w.state.position


# with one particle more the density pass has one lane per particle; h of 0.02 edges, or every
# particle NaN (all of them in one voxel, no pair within h)
@pytest.mark.parametrize("form", ["coarse", "nan"])
def test_a_crowd_costs_no_more_than_with_one_lane(gpu, form):
    def density_ms(n):
        h = 0.4 * (30 / (4.0 / 3.0 * np.pi * n)) ** (1.0 / 3.0)
        s, pos = strategy(n, h, 0.02 if form == "coarse" else 0.3, gpu)
        if form == "nan":
            pos = np.full_like(pos, np.nan)
        rows = [torch.from_numpy(np.ascontiguousarray(pos[:, d], dtype=np.float32)).to(gpu) for d in range(3)]
        got = []
        for _ in range(3):
            s.ctx.upload_f32(*rows, *[torch.zeros_like(r) for r in rows])
            got.append(s.ctx.step_timed(1)["density"])
        return float(np.median(got))

    assert density_ms(MOST) <= 1.3 * density_ms(MOST + 1)


# 0.15 and 0.04 edges are where the limits change
@pytest.mark.parametrize("n,edges", [(131072, 0.14), (131073, 0.14), (98304, 0.03), (98305, 0.03), (20011, 0.1), (1500, 0.05)])
def test_coarse_voxels_equal_one_lane(gpu, n, edges):
    h = (30 / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0)
    s, pos = strategy(MOST + 1, h, edges, gpu)
    rng = np.random.default_rng(142)
    vel = rng.normal(0.0, 0.3, size=(MOST + 1, 3))
    pos[n:] = rng.uniform(0.7, 0.95, size=(MOST + 1 - n, 3))
    # the others' voxels may hold the first n particles' too: those come first in each, by their ids
    want = s.advance(SimulationState(pos, vel, np.zeros(MOST + 1)), 1)
    got = strategy(n, h, edges, gpu)[0].advance(SimulationState(pos[:n], vel[:n], np.zeros(n)), 1)
    for f in ("position", "velocity", "density"):
        assert np.array_equal(getattr(got, f), getattr(want, f)[:n], equal_nan=True), f
