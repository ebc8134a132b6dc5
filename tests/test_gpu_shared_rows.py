"""16 lanes per particle: the four particles of a wavefront search dense surroundings together."""
import numpy as np
import pytest

import oracle
from _brute import naive_terms
from sph_amd import BatchedSPH, NaiveSPHStrategy
from sph_amd.data_classes import SimulationState
from sph_amd.workloads import box_uniform, voxel_for

pytestmark = pytest.mark.gpu

TOL = 1e-5  # of the density and of the sum of the pair terms' magnitudes, as for the other lane counts


# neighbours around and well past the 192 that a list and its tail serve (at the box's faces fewer:
# wavefronts of both kinds); a last wavefront that is not full; whole cells; more than 64 rows
# (scale 0.25); two clusters, whose seam lies inside a wavefront
@pytest.mark.parametrize("n,mean,scale,slabs,clusters", [
    (3, 30, 1.0, True, 1), (1603, 300, 1.0, True, 1), (2999, 700, 0.5, True, 1), (1501, 800, 1.0, False, 1),
    (2003, 400, 0.25, True, 1), (2001, 500, 0.5, True, 2)])
def test_shared_rows_match_oracle(gpu, n, mean, scale, slabs, clusters):
    h = min(0.3, (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0))
    w = box_uniform(n, seed=91, h=h)
    rng = np.random.default_rng(92)
    pos = w.state.position
    if clusters == 2:
        pos[n // 2 + 1:] += 0.4
    pos = pos.astype(np.float32).astype(np.float64)
    vel = rng.normal(0.0, 0.3, size=(n, 3)).astype(np.float32).astype(np.float64)
    state = SimulationState(pos, vel, np.zeros(n))
    strat = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu, grid_voxel=voxel_for(h) * scale, lanes=16,
                             slabs=slabs, keep_terms=True)
    out = strat.compute_next_state(state)
    _, _, rho, force, _ = oracle.step(pos, vel, consts=w.constants, ext=w.params.external_force, dt=1.0 / w.params.fps,
                                      space=w.params.space_size, voxel=w.params.voxel_size, mode="BOX",
                                      formulation="NAIVE", pipe=None, rng=None)
    assert np.max(np.abs(out.density - rho) / rho) <= TOL
    _, _, _, sp, sv = naive_terms(pos, vel, w.constants)
    assert np.max(np.linalg.norm(strat.result_force - force, axis=1) / np.maximum(sp + sv, 1e-30)) <= TOL
    if slabs:
        batch = BatchedSPH([(w.params, w.constants)], device=gpu, cell_scale=[scale], lanes=[16])
        batch.upload([state])
        batch.step(1)
        got = batch.download()[0]
        for f in ("position", "velocity", "density"):
            assert np.array_equal(getattr(got, f), getattr(out, f)), f
