"""Scans of all candidates, past the 192 neighbours that a list and its tail serve, by few lanes."""
import numpy as np
import pytest
import torch

import oracle
from _brute import naive_terms
from sph_amd import NaiveSPHStrategy
from sph_amd.data_classes import SimulationState
from sph_amd.workloads import box_uniform, voxel_for

pytestmark = pytest.mark.gpu

TOL = 1e-5  # of the density and of the sum of the pair terms' magnitudes, as for the other lane counts


def case(n, mean, seed):
    h = min(0.3, (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0))
    return box_uniform(n, seed=seed, h=h), voxel_for(h)


# rows of a few candidates (cells of h / 4) and of hundreds, which end at every place of a load of two
# or three batches
@pytest.mark.parametrize("lanes", [2, 4, 8])
@pytest.mark.parametrize("n,mean,scale", [(211, 200, 0.25), (1501, 250, 0.5), (2003, 600, 1.0)])
def test_scans_match_oracle(gpu, lanes, n, mean, scale):
    w, voxel = case(n, mean, 181)
    pos = w.state.position.astype(np.float32).astype(np.float64)
    vel = np.random.default_rng(182).normal(0.0, 0.3, size=(n, 3)).astype(np.float32).astype(np.float64)
    strat = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu, grid_voxel=voxel * scale, lanes=lanes,
                             keep_terms=True)
    out = strat.compute_next_state(SimulationState(pos, vel, np.zeros(n)))
    _, _, rho, force, _ = oracle.step(pos, vel, consts=w.constants, ext=w.params.external_force, dt=1.0 / w.params.fps,
                                      space=w.params.space_size, voxel=w.params.voxel_size, mode="BOX",
                                      formulation="NAIVE", pipe=None, rng=None)
    assert np.max(np.abs(out.density - rho) / rho) <= TOL
    _, _, _, sp, sv = naive_terms(pos, vel, w.constants)
    assert np.max(np.linalg.norm(strat.result_force - force, axis=1) / np.maximum(sp + sv, 1e-30)) <= TOL


def test_a_scan_by_two_lanes(gpu):
    """The force pass scans the candidates that the density pass scanned: 0.99 of its time before the scan
    looked one batch ahead, 1.23 while it did, 0.93 with three batches at once."""
    w, _ = case(4099, 300, 183)
    s = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu, lanes=2, check_finite=False)
    rows = [torch.from_numpy(np.ascontiguousarray(w.state.position[:, d], dtype=np.float32)).to(gpu) for d in range(3)]
    got = []
    for _ in range(9):
        s.ctx.upload_f32(*rows, *[torch.zeros_like(r) for r in rows])
        s.ctx.step(1)
        ms = s.ctx.step_timed(4)
        got.append(ms["force"] / ms["density"])
    assert np.median(got) <= 1.1
