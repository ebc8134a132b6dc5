"""The VOXEL formulation's sort and cell table against the host's order."""
import numpy as np
import pytest
import torch

from sph_amd import _native as N
from sph_amd.constants import SPHConstants
from sph_amd.data_classes import SimulationParameters
from sph_amd.strategy import VoxelSPHStrategy
from sph_amd.workloads import box_uniform

pytestmark = pytest.mark.gpu


# tiles of 512 keys whose counts the downsweep adds up to 49,152 particles, with the scan to 196,608,
# of 1,024 to 786,432 and of 2,048 from there; the corner boxes leave long runs of empty cells
# before and after them (tables of 4,096 cells, of a multiple of that and of 35,937)
@pytest.mark.parametrize("n,low,high,edge", [
    (1, 0.5, 0.6, 16), (511, 0.0, 1.0, 16), (513, 0.9, 1.0, 64), (4097, 0.4, 0.5, 33), (49152, 0.0, 0.3, 64),
    (49153, 0.6, 1.0, 64), (196608, 0.0, 1.0, 33), (196609, 0.0, 0.2, 64), (786432, 0.0, 1.0, 64), (786433, 0.3, 0.7, 64)])
def test_order_and_table(gpu, n, low, high, edge):
    voxel = np.float32(1.0 / edge)
    p = SimulationParameters(n, np.array([0.0, -9.81, 0.0]), 1, 1000, box_uniform(16).params.pipe, np.ones(3),
                             np.array([voxel] * 3, dtype=np.float64))
    c = SPHConstants(h=float(voxel), mass=0.02, rho0=1000.0, k=3.0, visc=3.5, damp=0.5)
    s = VoxelSPHStrategy(p, constants=c, device=gpu, check_finite=False)
    dims = s.voxel_dims
    rng = np.random.default_rng(111)
    cell = rng.integers(int(low * edge), max(int(high * edge), int(low * edge) + 1), size=(n, 3))
    pos = ((cell + rng.uniform(0.1, 0.9, size=(n, 3))) * voxel).astype(np.float32)  # clear of the bounds
    key = cell[:, 0] + dims[0] * (cell[:, 1] + dims[1] * cell[:, 2])
    want = np.argsort(key, kind="stable")
    begin = np.full(int(np.prod(dims)), -1)
    ks, first = np.unique(key[want], return_index=True)
    begin[ks] = first
    rows = [torch.from_numpy(np.ascontiguousarray(pos[:, d])).to(gpu) for d in range(3)]
    zero = torch.zeros_like(rows[0])

    def check():
        assert np.array_equal(s.ctx.read_buffer(N.BUF_PERM).cpu().numpy(), want)
        assert np.array_equal(s.ctx.read_buffer(N.BUF_CELL_BEGIN).cpu().numpy(), begin)
        assert np.array_equal(s.ctx.read_buffer(N.BUF_SORTED_KEYS).cpu().numpy(), key[want])

    s.ctx.upload_f32(*rows, *[zero] * 3)
    s.ctx.step(1)
    check()
    s.ctx.upload_f32(*rows, *[zero] * 3)
    s.ctx.run_stage(N.STAGE_SORT)
    s.ctx.run_stage(N.STAGE_TABLE)
    check()
