"""Neighbour sets, seen through sums that a single missing or doubled neighbour changes."""
import numpy as np
import pytest
import torch

from sph_amd import BatchedSPH, NaiveSPHStrategy
from sph_amd.constants import SPHConstants
from sph_amd.data_classes import SimulationParameters, SimulationState
from sph_amd.workloads import box_uniform

pytestmark = pytest.mark.gpu

H = 0.0625


def parameters(n, voxel):
    p = SimulationParameters(n, np.array([0.0, -9.81, 0.0]), 1, 10000, box_uniform(16).params.pipe, np.ones(3),
                             np.array([voxel] * 3))
    return p, SPHConstants(h=H, mass=0.02, rho0=1000.0, k=3.0, visc=3.5, damp=0.5)


# Positions on a lattice of h / 4: r^2 / h^2 is a multiple of 1/16, a term (1 - r^2 / h^2)^3 of 2^-12, and a
# sum of up to 2,800 terms fits 24 bits, so it is exact in any order and misses no neighbour closer
# than h.  per: particles of a lattice place (257 places lie within h), 0.05 to 10: 12 to 2,600
# neighbours.  scale: cells of h, h / 2 and h / 4 (9, 25 and 81 rows)
@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("n,per,scale", [(1, 1, 1.0), (31, 0.2, 0.5), (3001, 0.05, 0.5), (3001, 0.12, 1.0), (3001, 0.43, 0.25),
                                         (3001, 1, 0.5), (6007, 10, 1.0), (6007, 3, 0.25), (120001, 1, 1.0)])
def test_exact_sums(gpu, lanes, n, per, scale):
    rng = np.random.default_rng(121)
    side = int(np.ceil((n / per) ** (1.0 / 3.0)))
    site = rng.permutation(np.repeat(np.arange(side ** 3), int(np.ceil(per))))[:n]
    at = np.stack([site % side, site // side % side, site // side ** 2], axis=1)
    assert side <= 56
    pos = torch.from_numpy(at * (H / 4) + 0.0625)  # exact in FP32
    count = torch.zeros((side + 8,) * 3, dtype=torch.float64)
    count.index_put_(tuple(torch.from_numpy(at.T) + 4), torch.ones(n, dtype=torch.float64), accumulate=True)
    d2 = (torch.arange(-4, 5) ** 2).double()
    kernel = (1.0 - (d2[:, None, None] + d2[None, :, None] + d2[None, None, :]) / 16.0).clamp(min=0.0) ** 3
    sums = torch.nn.functional.conv3d(count[None, None], kernel[None, None])[0, 0][tuple(torch.from_numpy(at.T))]
    assert float(sums.max()) < 4096.0
    p, c = parameters(n, H * scale)
    state = SimulationState(pos.numpy(), np.zeros((n, 3)), np.zeros(n))
    # the factor of the sum as the step holds it, and one rounding of the product
    factor = np.float32(c.mass * 315.0 / (64.0 * np.pi * H ** 3))
    want = (factor * sums.numpy().astype(np.float32)).astype(np.float64)
    got = NaiveSPHStrategy(p, constants=c, device=gpu, lanes=lanes, check_finite=False).compute_next_state(state)
    assert np.array_equal(got.density, want)
    batch = BatchedSPH([(p, c)], device=gpu, lanes=[lanes])
    batch.upload([state])
    batch.step(1)
    assert np.array_equal(batch.download()[0].density, want)


# one cell of 700 (ordered through the bitmap) with few particles in its lower slabs, so that its
# table entry keeps their offsets; the neighbours in the cells around it stop and start at them
@pytest.mark.parametrize("lower", [(1, 0, 0), (2, 3, 1), (0, 0, 6), (0, 7, 0)])
def test_slab_offsets_of_a_heavy_cell(gpu, lower):
    rng = np.random.default_rng(122)
    n, voxel, many = 6000, 0.125, 73729  # past the sort in one launch
    pos = rng.uniform(0.0, 0.5, size=(n, 3))
    heavy = np.all(np.floor(pos / voxel) == 1, axis=1)
    pos[heavy, 0] += voxel  # the cell holds nothing but what follows
    cell = np.concatenate([rng.uniform(1 + q / 4, 1 + (q + 1) / 4, size=k) for q, k in enumerate((*lower, 700 - sum(lower)))])
    pos[:700, 0] = voxel * cell
    pos[:700, 1:] = rng.uniform(voxel, 2 * voxel, size=(700, 2))
    pos[700:] = pos[700:][rng.permutation(n - 700)]
    pos = pos.astype(np.float32)
    slab = np.floor(pos[:, 0] / voxel * 4).astype(int) - 4
    inside = np.all(np.floor(pos / voxel) == 1, axis=1)
    counts = [int(np.sum(inside & (slab == q))) for q in range(4)]
    assert counts[:3] == list(lower) and sum(counts) == 700
    far = rng.uniform(0.75, 1.0, size=(many - n, 3)).astype(np.float32)
    got = []
    for p in (pos, np.concatenate([pos, far])):
        par, c = parameters(len(p), voxel)
        s = NaiveSPHStrategy(par, constants=SPHConstants(h=0.1, mass=c.mass, rho0=c.rho0, k=c.k, visc=c.visc, damp=c.damp),
                             device=gpu, check_finite=False)
        rows = [torch.from_numpy(np.ascontiguousarray(p[:, d])).to(gpu) for d in range(3)]
        s.ctx.upload_f32(*rows, *[torch.zeros_like(r) for r in rows])
        s.ctx.step(1)
        got.append([t[:n].cpu().numpy() for t in s.ctx.download_f32()])
    for a, b in zip(*got):  # both sum in the same order
        assert np.array_equal(a, b)
