"""Large problems: neighbour lists beyond the int16 window of a particle's own index."""
import numpy as np
import pytest
import torch

import oracle
from sph_amd import _native as N
from sph_amd.constants import SPHConstants
from sph_amd.data_classes import SimulationParameters, SimulationState
from sph_amd.strategy import NaiveSPHStrategy
from sph_amd.workloads import box_uniform

pytestmark = pytest.mark.gpu

TOL = 1e-5  # as in test_gpu_step.py
MANY = 1 << 20  # up to here the one-lane density pass keeps to the int16 window


def slab(n, layers, seed=71):
    """n particles, about 30 neighbours each, in a slab of `layers` cell layers in z: two
    layers are n / layers particles apart in cell order."""
    h, vx = 0.0457, 0.03125
    edge = (n / (30.0 / (4.0 / 3.0 * np.pi * h ** 3)) / (layers * vx)) ** 0.5
    rng = np.random.default_rng(seed)
    space = np.array([edge, edge, layers * vx])
    f32 = lambda a: a.astype(np.float32).astype(np.float64)  # noqa: E731
    pos, vel = f32(rng.uniform(0.0, 1.0, size=(n, 3)) * space), f32(rng.normal(0.0, 0.1, size=(n, 3)))
    pos = np.minimum(pos, f32(space) * (1 - 1e-6))
    c = SPHConstants(h=h, mass=0.02, rho0=1000.0, k=3.0, visc=3.5, damp=0.5)
    p = SimulationParameters(n, np.array([0.0, -9.81, 0.0]), 1, 1000, box_uniform(16).params.pipe, space,
                             np.array([vx, vx, vx]))
    return p, c, pos, vel


# layers 41: 25,600 slots to the next layer, past the window two layers on; 20: 52,000, past the
# window, within reach of the lists; 10: 105,000, beyond their reach (rescanned)
@pytest.mark.parametrize("n,layers", [(MANY, 20), (MANY + 1, 41), (MANY + 77, 20), (MANY + 77, 10)])
def test_lists_beyond_the_window(gpu, n, layers):
    p, c, pos, vel = slab(n, layers)
    strat = NaiveSPHStrategy(p, constants=c, device=gpu)
    out = strat.compute_next_state(SimulationState(pos, vel, np.zeros(n)))
    rp, _, rrho, _, _ = oracle.step(pos, vel, consts=c, ext=p.external_force, dt=1e-3, space=p.space_size,
                                    voxel=p.voxel_size, use_grid=True)
    drho = np.abs(out.density - rrho) / rrho
    dpos = np.abs(out.position - rp) / np.maximum(np.abs(rp), 1e-3)
    # a coordinate that ends within FP32 rounding of a wall may count as past it on one side only:
    # there the one result is the wall itself, to rounding, and the other the place 1e-3 inside it
    for wall, inside in ((0.0, 1e-3), (p.space_size, p.space_size - 1e-3)):
        for one, other in ((out.position, rp), (rp, out.position)):
            dpos[(np.abs(one - wall) <= 1e-6) & (np.abs(other - inside) <= 1e-6)] = 0.0
    print(f"n {n} layers {layers}: rho {drho.max():.2e} pos {dpos.max():.2e}")
    assert drho.max() <= TOL and dpos.max() <= TOL


def test_pullback_from_far_lists(gpu):
    """A snapshot whose lists reach beyond the window, reversed with the lanes it was made with
    (which walk the lists) and with two (which cannot decode them, and scan the candidates)."""
    n = MANY + 77
    p, c, pos, vel = slab(n, 20)
    par = N.make_params(n, p.external_force, 1e-3, p.space_size, p.voxel_size, N.SPH_MODE_BOX, N.SPH_FORM_NAIVE,
                        flags=N.SPH_FLAG_ADJOINT)
    ctx = N.NativeContext(par, N.make_consts(c), gpu)
    rows = [torch.from_numpy(np.ascontiguousarray(a[:, k], dtype=np.float32)).to(gpu) for a in (pos, vel) for k in range(3)]
    ctx.upload_f32(*rows)
    snap = torch.empty(ctx.adjoint_snapshot_bytes(), dtype=torch.uint8, device=gpu)
    ctx.step_save(snap)
    g = torch.from_numpy(np.random.default_rng(72).normal(size=(2, n, 3)).astype(np.float32)).to(gpu)
    got = []
    for lanes in (1, 2):
        ctx.set_lanes(lanes)
        ctx.adjoint_seed(g[0], g[1])
        ctx.adjoint_step_from(snap)
        got.append([t.double() for t in ctx.adjoint_read()])
    for a, b in zip(*got):
        assert float((a - b).norm() / b.norm()) <= TOL


# 96 list slots; up to 192 neighbours the force pass walks the list and then the candidates after
# its last neighbour, past that it scans all candidates.  h sets the mean: 60, 97, 150 and 250.
@pytest.mark.parametrize("lanes", [1, 2, 8, 64])
@pytest.mark.parametrize("mean", [60, 97, 150, 250])
def test_lists_past_their_slots(gpu, mean, lanes):
    n = 3001
    h = (mean / (n / 0.4 ** 3) / (4.0 / 3.0 * np.pi)) ** (1.0 / 3.0)
    w = box_uniform(n, seed=73, h=h)
    rng = np.random.default_rng(74)
    pos = w.state.position.astype(np.float32).astype(np.float64)
    vel = rng.normal(0.0, 0.3, size=(n, 3)).astype(np.float32).astype(np.float64)
    strat = NaiveSPHStrategy(w.params, constants=w.constants, device=gpu, lanes=lanes)
    out = strat.compute_next_state(SimulationState(pos, vel, np.zeros(n)))
    rp, rv, rrho, _, _ = oracle.step(pos, vel, consts=w.constants, ext=w.params.external_force, dt=1e-3,
                                     space=w.params.space_size, voxel=w.params.voxel_size)
    assert (np.abs(out.density - rrho) / rrho).max() <= TOL
    assert (np.abs(out.position - rp) / np.maximum(np.abs(rp), 1e-3)).max() <= TOL
    assert np.abs(out.velocity - rv).max() / np.abs(rv).max() <= TOL
