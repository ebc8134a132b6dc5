"""The one-launch sort of few particles where they crowd into few cells or a few layers of them."""
import numpy as np
import pytest
import torch

from sph_amd import NaiveSPHStrategy
from sph_amd import _native as N
from sph_amd.constants import SPHConstants
from sph_amd.data_classes import SimulationParameters
from sph_amd.workloads import box_uniform

pytestmark = pytest.mark.gpu

ONE = 73728  # the largest count the one-launch sort takes
VOXEL = 0.015625


def context(n, space, h, gpu, slabs=True, lanes=8):
    p = SimulationParameters(n, np.array([0.0, -9.81, 0.0]), 1, 10000, box_uniform(16).params.pipe, np.asarray(space),
                             np.array([VOXEL] * 3))
    c = SPHConstants(h=h, mass=0.02, rho0=1000.0, k=3.0, visc=3.5, damp=0.5)
    return NaiveSPHStrategy(p, constants=c, device=gpu, check_finite=False, slabs=slabs, lanes=lanes)


def rows(pos, gpu):
    r = [torch.from_numpy(np.ascontiguousarray(pos[:, d], dtype=np.float32)).to(gpu) for d in range(3)]
    return [*r, *[torch.zeros_like(r[0])] * 3]


def crowd(n, per, space, seed, ordered):
    """n particles, about `per` in each of the first cells of the lowest layer."""
    rng = np.random.default_rng(seed)
    cells = -(-n // per)
    nx = min(cells, int(space[0] / VOXEL))
    size = np.array([nx * VOXEL, -(-cells // nx) * VOXEL, VOXEL])
    pos = (rng.uniform(0.0, 1.0, size=(n, 3)) * size).astype(np.float32)
    if ordered:  # slots nearly in cell order, as between the steps of a run
        pos = pos[np.lexsort((pos[:, 0], np.floor(pos[:, 1] / VOXEL)))]
    return pos


# 1,024 is the fewest particles for which ranges are shared; 5 x 5 x 9 cells give ranges of 2, the last
# with one; 500 in a cell stay below the bitmap, 600 do not; a background leaves a particle here and
# there in the other ranges; 300 in each of three cells: more parts than cells
@pytest.mark.parametrize("n,per,space,background", [
    (1023, 30, (1.0, 1.0, 0.25), 0), (1024, 30, (1.0, 1.0, 0.25), 10), (4099, 40, (5 * VOXEL, 5 * VOXEL, 9 * VOXEL), 900),
    (1500, 500, (1.0, 1.0, 1.0), 0), (20011, 100, (1.0, 1.0, 1.0), 3000), (65537, 500, (4.0, 1.0, 1.0), 0),
    (ONE, 30, (4.0, 1.0, 1.0), 500), (ONE, 600, (1.0, 1.0, 1.0), 5000), (ONE, ONE // 3 + 1, (1.0, 1.0, 1.0), 100),
    (30001, 9000, (1.0, 1.0, 0.5), 0)])
@pytest.mark.parametrize("slabs,ordered", [(True, False), (True, True), (False, True)])
def test_crowds_are_ordered(gpu, n, per, space, background, slabs, ordered):
    pos = crowd(n, per, space, 111, ordered)
    rng = np.random.default_rng(112)
    pos[rng.choice(n, background, replace=False)] = (rng.uniform(0.0, 1.0, size=(background, 3)) * space).astype(np.float32)
    s = context(n, space, 0.004, gpu, slabs=slabs)
    dims = s.voxel_dims
    cell = np.clip(np.floor(pos / np.float32(VOXEL)).astype(np.int64), 0, np.asarray(dims) - 1)
    key = cell[:, 0] + dims[0] * (cell[:, 1] + dims[1] * cell[:, 2])
    slab = np.clip(np.floor(pos[:, 0].astype(np.float64) / VOXEL * 4) - 4 * cell[:, 0], 0, 3).astype(np.int64)
    begin = np.full(int(np.prod(dims)), -1)
    ks, first = np.unique(np.sort(key), return_index=True)
    begin[ks] = first
    state = rows(pos, gpu)
    for staged in (False, True):
        s.ctx.upload_f32(*state)
        if staged:  # (cell, id)
            s.ctx.run_stage(N.STAGE_SORT)
            want = np.lexsort((np.arange(n), key))
        else:  # (cell, slab, id)
            s.ctx.step(1)
            want = np.lexsort((np.arange(n), slab if slabs else np.zeros(n), key))
        assert np.array_equal(s.ctx.read_buffer(N.BUF_PERM).cpu().numpy(), want)
        if staged:
            s.ctx.run_stage(N.STAGE_TABLE)
        assert np.array_equal(s.ctx.read_buffer(N.BUF_CELL_BEGIN).cpu().numpy(), begin)
        assert np.array_equal(s.ctx.read_buffer(N.BUF_SORTED_KEYS).cpu().numpy(), key[want])


@pytest.mark.parametrize("per", [30, 100, 500])
def test_a_crowd_costs_no_more_than_in_several_launches(gpu, per):
    """65,537 particles in a row of cells at the bottom of 1,048,576, once by themselves and once with
    8,192 more far away, which take them past the one-launch sort: a workgroup that sorts the crowd alone
    takes 10 to 40 times as long as those launches."""
    n, space = 65537, (1.0, 1.0, 4.0)
    pos = crowd(n, per, space, 113, False)
    far = (np.random.default_rng(114).uniform(0.5, 1.0, size=(ONE + 1 - n, 3)) * space).astype(np.float32)

    def sort_ms(p):
        s, state, got = context(len(p), space, VOXEL / 4, gpu), rows(p, gpu), []
        for _ in range(5):
            s.ctx.upload_f32(*state)
            s.ctx.step(1)
            got.append(s.ctx.step_timed(4)["sort"])
        return float(np.median(got))

    assert sort_ms(pos) <= 2.0 * sort_ms(np.concatenate([pos, far]))
