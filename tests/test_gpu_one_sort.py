"""The one-launch sort of few particles against the host's order: cells, slabs, ids and tables."""
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


def context(n, voxel, h, gpu, space=(1.0, 1.0, 1.0), slabs=True):
    p = SimulationParameters(n, np.array([0.0, -9.81, 0.0]), 1, 1000, box_uniform(16).params.pipe, np.asarray(space),
                             np.array([voxel] * 3))
    c = SPHConstants(h=h, mass=0.02, rho0=1000.0, k=3.0, visc=3.5, damp=0.5)
    return NaiveSPHStrategy(p, constants=c, device=gpu, check_finite=False, slabs=slabs)


def expected(pos, voxel, dims):
    cell = np.clip(np.floor(pos / voxel).astype(np.int64), 0, np.asarray(dims) - 1)
    key = cell[:, 0] + dims[0] * (cell[:, 1] + dims[1] * cell[:, 2])
    slab = np.clip(np.floor(pos[:, 0].astype(np.float64) / voxel * 4) - 4 * cell[:, 0], 0, 3).astype(np.int64)
    return key, slab


# uniform; everything in a tenth of the box (a range's list in global memory); one cell of 600 and
# of all particles (ordered through the bitmap); one particle; the largest count and the next
@pytest.mark.parametrize("n,spread,heavy,voxel", [
    (1, 1.0, 0, 0.0625), (5, 1.0, 0, 0.0625), (4096, 1.0, 0, 0.0625), (4099, 1.0, 600, 0.125), (30001, 0.1, 0, 0.03125),
    (9000, 0.001, 0, 0.0625), (20000, 1.0, 20000, 0.25), (ONE, 0.4, 700, 0.015625), (ONE + 1, 0.4, 700, 0.015625)])
@pytest.mark.parametrize("slabs", [True, False])
def test_order_and_table(gpu, n, spread, heavy, voxel, slabs):
    rng = np.random.default_rng(101)
    pos = rng.uniform(0.0, spread, size=(n, 3))
    pos[:heavy] = rng.uniform(voxel, 2 * voxel, size=(heavy, 3))  # all in cell (1, 1, 1)
    pos = rng.permutation(pos).astype(np.float32)
    s = context(n, voxel, 0.01, gpu, slabs=slabs)
    rows = [torch.from_numpy(np.ascontiguousarray(pos[:, d])).to(gpu) for d in range(3)]
    dims = s.voxel_dims
    key, slab = expected(pos, np.float32(voxel), dims)
    s.ctx.upload_f32(*rows, *[torch.zeros_like(r) for r in rows])
    s.ctx.step(1)  # the fused order: (cell, slab, id)
    perm = s.ctx.read_buffer(N.BUF_PERM).cpu().numpy()
    want = np.lexsort((np.arange(n), slab if slabs else np.zeros(n), key))
    assert np.array_equal(perm, want)
    begin = np.full(int(np.prod(dims)), -1)
    ks, first = np.unique(key[want], return_index=True)
    begin[ks] = first
    assert np.array_equal(s.ctx.read_buffer(N.BUF_CELL_BEGIN).cpu().numpy(), begin)
    assert np.array_equal(s.ctx.read_buffer(N.BUF_SORTED_KEYS).cpu().numpy(), key[want])
    s.ctx.upload_f32(*rows, *[torch.zeros_like(r) for r in rows])
    s.ctx.run_stage(N.STAGE_SORT)  # the staged order: (cell, id)
    want = np.lexsort((np.arange(n), key))
    assert np.array_equal(s.ctx.read_buffer(N.BUF_PERM).cpu().numpy(), want)
    s.ctx.run_stage(N.STAGE_TABLE)
    assert np.array_equal(s.ctx.read_buffer(N.BUF_CELL_BEGIN).cpu().numpy(), begin)


def test_neighbours_around_a_heavy_cell(gpu):
    """The slab offsets and counts that the heavy cell's table entry carries search the same
    pairs as the several-launch sort's: one density pass each, from a table of either."""
    n, voxel = 6000, 0.125
    rng = np.random.default_rng(102)
    pos = rng.uniform(0.0, 1.0, size=(n, 3))
    pos[:600, 0] = rng.uniform(voxel * 1.9, 2 * voxel, size=600)  # few below slab 3: offsets kept
    pos[:600, 1:] = rng.uniform(voxel, 2 * voxel, size=(600, 2))
    pos = pos.astype(np.float32)
    rows = [torch.from_numpy(np.ascontiguousarray(pos[:, d])).to(gpu) for d in range(3)]
    got = []
    for slabs in (True, False):
        s = context(n, voxel, 0.1, gpu, slabs=slabs)
        s.ctx.upload_f32(*rows, *[torch.zeros_like(r) for r in rows])
        s.ctx.step(1)
        got.append(s.ctx.download_f32()[6].double())
    assert float(((got[0] - got[1]).abs() / got[1]).max()) <= 1e-5


# 256 ranges of 4,096 cells, the most the one-launch sort takes, and one layer of cells more
@pytest.mark.parametrize("depth", [64, 65])
def test_most_cells(gpu, depth):
    n, voxel = 70001, 0.015625
    space = (4.0, 1.0, depth * voxel)
    pos = (np.random.default_rng(103).uniform(0.0, 1.0, size=(n, 3)) * space).astype(np.float32)
    s = context(n, voxel, 0.01, gpu, space=space)
    key, slab = expected(pos, np.float32(voxel), s.voxel_dims)
    rows = [torch.from_numpy(np.ascontiguousarray(pos[:, d])).to(gpu) for d in range(3)]
    s.ctx.upload_f32(*rows, *[torch.zeros_like(r) for r in rows])
    s.ctx.step(1)
    want = np.lexsort((np.arange(n), slab, key))
    assert np.array_equal(s.ctx.read_buffer(N.BUF_PERM).cpu().numpy(), want)
