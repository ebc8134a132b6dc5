"""Timed cases of the SPH step: the calls a user's program makes, over the sizes it makes them at.

A case is a dict of plain values.  Its "kind" is the kind of program:

  frames     the reference's frame loop: compute_next_state() on host arrays, every frame kept.
             The strategy has its default settings, the first frame uploads the state, the
             following ones pass the returned state back.  Frames are recorded as FP32, which
             is what their values are.
  steps      a program that holds its state on the device: upload, a few steps (launched one by
             one, or replayed as a HIP graph recorded beforehand), download, all FP32.
  batch      many simulations of uneven sizes in one context, as "steps".
  gradients  a differentiable rollout: the loss on its final state, and the gradients with
             respect to the initial positions, the initial velocities and the viscosity.

and its "flow" what is simulated: "box" (particles uniform in [0.1, 0.5]^3 of the unit box),
"dam" (the jittered lattice of the dam break), "pipe" (the 8-segment pipe), "reference_box" and
"reference_pipe" (the reference's own run configuration).  The steps of a pass are few, so that
a rounding difference does not grow into another trajectory (a wall hit one step earlier).
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "cuda-sph_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "cuda-sph_amd"))


def listed():
    return [
        # the reference's CPU-sized case in its frame loop: latency of the whole call
        dict(name="frames_box_4k", kind="frames", flow="box", formulation="NAIVE", n=4096, h=0.0457, steps=3),
        # the reference's default run (20,000 particles, h = 2, about 105 neighbours) in a box
        dict(name="frames_reference_box", kind="frames", flow="reference_box", formulation="NAIVE", n=20000, steps=2),
        # the same with the VOXEL formulation, whose 32 list places are full there; one frame, since
        # the second finds particles that its forces have thrown far out of the box
        dict(name="frames_reference_voxel", kind="frames", flow="reference_box", formulation="VOXEL", n=20000, steps=1),
        # the CPU-sized case as the autotuner sets it up, held on the device, one graph launch
        dict(name="steps_box_4k", kind="steps", flow="box", formulation="NAIVE", n=4096, h=0.0457, steps=20, lanes=32,
             cell_scale=2.0, slabs=False, graph=True),
        # a mid-sized box of an odd particle count with the lanes the autotuner gives such sizes
        dict(name="steps_box_65537", kind="steps", flow="box", formulation="NAIVE", n=65537, h=0.0, steps=8, lanes=4,
             cell_scale=1.0, slabs=True, graph=False),
        # a ragged dam break between the small and the headline size
        dict(name="steps_dam_37x61x53", kind="steps", flow="dam", formulation="NAIVE", nx=37, ny=61, nz=53, steps=3,
             lanes=1, cell_scale=1.0, slabs=True, graph=False),
        # the headline workload: 1,048,576 particles
        dict(name="steps_dam_1m", kind="steps", flow="dam", formulation="NAIVE", nx=64, ny=128, nz=128, steps=3,
             lanes=1, cell_scale=1.0, slabs=True, graph=False),
        # the largest: 4.2 million particles, whose working set is beyond the caches
        dict(name="steps_dam_4m", kind="steps", flow="dam", formulation="NAIVE", nx=128, ny=192, nz=171, steps=2,
             lanes=1, cell_scale=1.0, slabs=True, graph=False),
        # the reference's VOXEL formulation on the headline dam break
        dict(name="steps_dam_1m_voxel", kind="steps", flow="dam", formulation="VOXEL", nx=64, ny=128, nz=128, steps=2,
             lanes=1, cell_scale=2.0, slabs=False, graph=False),
        # the pipe workload
        dict(name="steps_pipe_512k", kind="steps", flow="pipe", formulation="NAIVE", n=524288, steps=3, lanes=1,
             cell_scale=1.0, slabs=True, graph=False),
        # 64 uneven simulations (8 to 2,200 neighbours per particle) per launch
        dict(name="batch_64", kind="batch", flow="box", count=64, n_lo=2048, n_hi=65536, steps=4, graph=True),
        # gradients of a rollout of the 16,384-particle box, forward and backward
        dict(name="gradients_16k", kind="gradients", flow="box", n=16384, h=0.0457, steps=20, every=20, lanes=32,
             keep_all=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _lanes_for(n):
    """About what the autotuner picks: lanes until the launch holds some 500,000 threads."""
    lanes = 1
    while lanes < 32 and n * lanes * 2 <= 1 << 19:
        lanes *= 2
    return lanes


def draw(rng: random.Random):
    kind = rng.choice(("frames", "frames", "steps", "steps", "steps", "batch", "gradients"))
    if kind == "frames":
        flow = rng.choice(("box", "reference_box", "reference_pipe"))
        c = dict(kind=kind, flow=flow, formulation="NAIVE", n=_log_int(rng, 1000, 50000), steps=rng.randint(1, 3))
        if flow == "box":
            c["h"] = 0.0
        # VOXEL where no particle is isolated (its density leaves the particle itself out)
        if flow == "reference_box" and c["n"] >= 12000:
            c.update(formulation="VOXEL", steps=1)
        return c
    if kind == "steps":
        flow = rng.choice(("box", "dam", "pipe"))
        c = dict(kind=kind, flow=flow, formulation="NAIVE", steps=rng.randint(1, 3), cell_scale=1.0, slabs=True,
                 graph=rng.random() < 0.3)
        if flow == "dam":
            c.update(nx=rng.randint(16, 80), ny=rng.randint(24, 150), nz=rng.randint(24, 150))
            n = c["nx"] * c["ny"] * c["nz"]
            if rng.random() < 0.35:
                c.update(formulation="VOXEL", cell_scale=2.0, slabs=False)
        else:
            n = c["n"] = _log_int(rng, 1500, 600000)
            if flow == "box":
                c["h"] = 0.0
        c["lanes"] = 1 if c["formulation"] == "VOXEL" else _lanes_for(n)
        return c
    if kind == "batch":
        return dict(kind=kind, flow="box", count=rng.randint(2, 40), n_lo=rng.randint(500, 2000),
                    n_hi=_log_int(rng, 4000, 40000), steps=rng.randint(1, 4), graph=rng.random() < 0.5)
    n = _log_int(rng, 2000, 40000)
    steps = rng.randint(4, 20)
    return dict(kind=kind, flow="box", n=n, h=0.0, steps=steps, every=rng.randint(2, steps), lanes=_lanes_for(n),
                keep_all=rng.random() < 0.6)


# ---------------------------------------------------------------------------------------
# Inputs: the workloads of the package, from the seed
# ---------------------------------------------------------------------------------------
def _box_h(case):
    """The case's h, or the one that gives about 30 neighbours."""
    return case["h"] or 0.4 * (30.0 / (4.0 / 3.0 * math.pi * case["n"])) ** (1.0 / 3.0)


def _workload(case, seed):
    """(params, constants, state, mode) of a single simulation."""
    from dataclasses import replace

    from sph_amd import initial_states, workloads

    flow = case["flow"]
    if flow in ("reference_box", "reference_pipe"):
        return initial_states.preset("BOX" if flow == "reference_box" else "PIPE", case["n"], seed)
    if flow == "box":
        w = workloads.box_uniform(case["n"], seed=seed, h=_box_h(case))
    elif flow == "dam":
        # in motion: from rest the pressures of the lattice nearly cancel, and what is left of
        # them is mostly rounding
        w = workloads.dam_break(case["nx"], case["ny"], case["nz"], seed=seed)
        vel = np.random.default_rng([seed, 5]).normal(0.0, 0.25, size=w.state.position.shape)
        w.state = replace(w.state, velocity=vel)
    else:
        w = workloads.pipe_flow(case["n"], seed=seed)
    scale = case.get("cell_scale", 1.0)
    if scale != 1.0:
        w.params = replace(w.params, voxel_size=np.asarray(w.params.voxel_size) * scale)
    return w.params, w.constants, w.state, w.mode


def _batch_instances(case, seed):
    from sph_amd import workloads

    # the instances' sizes, h, boxes and viscosities are the case's, their particles the seed's
    b = workloads.batch_64(seed=3, count=case["count"], steps=case["steps"], n_lo=case["n_lo"], n_hi=case["n_hi"])
    out = []
    for k, w in enumerate(b.instances):
        c = w.constants
        out.append(workloads.box_uniform(w.params.particle_count, seed=seed * 1000 + k, h=c.h, visc=c.visc,
                                         edge=float(w.params.space_size[0])))
    return out


def _batch_load(w):
    """Neighbours per particle of an instance: the rule the autotuner chooses lanes by."""
    edge = float(w.params.space_size[0])
    return w.params.particle_count / (0.4 * edge) ** 3 * 4.0 / 3.0 * math.pi * w.constants.h ** 3


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        from sph_amd import BatchedSPH

        inst = _batch_instances(case, seed)
        load = [_batch_load(w) for w in inst]
        batch = BatchedSPH([(w.params, w.constants) for w in inst],
                           cell_scale=[0.5 if x >= 2048 else 1.0 for x in load],
                           lanes=[min(16, max(1, 1 << int(math.log2(max(1.0, x / 32))))) for x in load])
        batch.upload([w.state for w in inst])
        pos, vel = batch.ctx_state_tensors()
        rows = torch.cat([pos.t(), vel.t()]).float().contiguous()
        return dict(case=case, ctx=batch.ctx, rows=rows, owner=batch,
                    graph=batch.capture(case["steps"]) if case["graph"] else None)
    params, consts, state, mode = _workload(case, seed)
    if kind == "frames":
        from sph_amd import make_strategy

        return dict(case=case, state=state,
                    strategy=make_strategy(case["formulation"], params, constants=consts, mode=mode))
    pos = torch.from_numpy(np.ascontiguousarray(state.position)).cuda().float()
    vel = torch.from_numpy(np.ascontiguousarray(state.velocity)).cuda().float()
    if kind == "gradients":
        from sph_amd import DifferentiableSPH

        sim = DifferentiableSPH(params, consts, steps=case["steps"], checkpoint_every=case["every"],
                                lanes=case["lanes"], keep_all=case["keep_all"])
        return dict(case=case, sim=sim, x0=pos.requires_grad_(), v0=vel.requires_grad_(),
                    mu=torch.tensor(consts.visc, requires_grad=True), target=_target(case, seed, pos.detach()))
    from sph_amd import make_strategy

    kw = {} if case["formulation"] == "VOXEL" else dict(lanes=case["lanes"], slabs=case["slabs"])
    strategy = make_strategy(case["formulation"], params, constants=consts, mode=mode, check_finite=False, **kw)
    rows = torch.cat([pos.t(), vel.t()]).contiguous()
    strategy.ctx.upload_f32(*rows)
    return dict(case=case, ctx=strategy.ctx, rows=rows, owner=strategy,
                graph=strategy.capture(case["steps"]) if case["graph"] else None)


def _target(case, seed, x0):
    """The positions a rollout is fitted to: the initial ones moved by about 1 cm."""
    noise = np.random.default_rng([seed, 44]).normal(0.0, 0.01, size=(case["n"], 3))
    return x0 + torch.from_numpy(noise.astype(np.float32)).to(x0.device)


# ---------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "frames":
        s, record = state["state"], []
        for _ in range(case["steps"]):
            s = state["strategy"].compute_next_state(s)
            record.append([a.astype(np.float32) for a in (s.position, s.velocity, s.density)])
        return record
    if kind == "gradients":
        from sph_amd import rollout

        x0, v0, mu = state["x0"], state["v0"], state["mu"]
        xT, vT = rollout(state["sim"], x0, v0, mu)
        loss = ((xT - state["target"]) ** 2).sum(1).mean()
        return [xT, vT, *torch.autograd.grad(loss, (x0, v0, mu))]
    ctx = state["ctx"]
    ctx.upload_f32(*state["rows"])
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        ctx.step(case["steps"])
    return ctx.download_f32()


def _pairs_estimate(case):
    """(particles, pairs within h) of one step, from the flow's mean number density."""
    def sphere(h):
        return 4.0 / 3.0 * math.pi * h ** 3

    if case["kind"] == "batch":
        inst = _batch_instances(case, 0)
        n = sum(w.params.particle_count for w in inst)
        return n, sum(w.params.particle_count * max(1.0, _batch_load(w)) for w in inst)
    if case["flow"] == "dam":
        n = case["nx"] * case["ny"] * case["nz"]
        return n, n * 30.0
    n = case["n"]
    if case["flow"] == "reference_box":
        per = n / (4.0 * 40.0 * 40.0) * sphere(2.0)
    elif case["flow"] == "reference_pipe":
        per = n / (40.0 * math.pi * 2.9 ** 2) * sphere(2.0)
    elif case["flow"] == "box":
        per = n / 0.064 * sphere(_box_h(case))
    else:
        per = 30.0
    if case.get("formulation") == "VOXEL":
        per = min(per, 32.0)
    return n, n * max(1.0, per)


def work(case):
    """Per step and particle 60 bytes (x, v and id read; x, v, id and rho written) and per pair
    11 operations for the density and 40 for the forces; beside that the states at the
    boundary.  A reversed step reads the step's state and the cotangent and writes the
    cotangent, and costs about 110 operations per pair."""
    n, pairs = _pairs_estimate(case)
    steps = case["steps"]
    if case["kind"] == "gradients":
        return {"bytes": n * (steps * (60 + 28 + 48 + 48) + 24 + 24 + 12 + 24), "flops": steps * pairs * (51 + 110)}
    boundary = 48 + steps * 56 if case["kind"] == "frames" else 24 + 28
    return {"bytes": n * (steps * 60 + boundary), "flops": steps * pairs * 51}


# ---------------------------------------------------------------------------------------
# The same in FP64, from the formulas
# ---------------------------------------------------------------------------------------
def _candidates(pos, edge, dims, ranges, step_rows):
    """For chunks of particles: (i, j) index pairs of every particle with the members of the
    cells around it, in the order of `ranges` (cell offsets; step_rows: each covers the cells
    -1 .. 1 along x) and of the particle number within a cell."""
    dev = pos.device
    d = torch.tensor(dims, device=dev)
    cell = torch.minimum((pos / edge).floor().long().clamp_(min=0), d - 1)
    key = cell[:, 0] + d[0] * (cell[:, 1] + d[1] * cell[:, 2])
    order = torch.sort(key, stable=True).indices
    count = torch.bincount(key, minlength=int(d.prod()))
    start = torch.cat([count.new_zeros(1), count.cumsum(0)])
    off = torch.tensor(ranges, device=dev)
    n, chunk = pos.shape[0], 1 << 17
    for a in range(0, n, chunk):
        c = cell[a:a + chunk, None, :] + off[None]
        inside = ((c[..., 1:] >= 0) & (c[..., 1:] < d[1:])).all(-1)
        row = d[0] * (c[..., 1] + d[1] * c[..., 2])
        if step_rows:
            lo, hi = (c[..., 0] - 1).clamp(min=0), torch.minimum(c[..., 0] + 1, d[0] - 1)
        else:
            lo = hi = c[..., 0]
            inside &= (lo >= 0) & (lo < d[0])
        first = torch.where(inside, start[(row + lo).clamp(0, count.numel() - 1)], 0)
        last = torch.where(inside, start[(row + hi).clamp(0, count.numel() - 1) + 1], 0)
        length, first = (last - first).reshape(-1), first.reshape(-1)
        end = length.cumsum(0)
        which = torch.repeat_interleave(torch.arange(length.numel(), device=dev), length)
        j = order[first[which] + torch.arange(which.numel(), device=dev) - (end - length)[which]]
        yield a, which // len(ranges) + a, j


def _pairs(x, case, consts, params):
    """(i, j) of the pairs the step sums over; VOXEL: the first 32 in its order, the particle
    itself counted among them."""
    h = consts.h
    out_i, out_j = [], []
    if case.get("formulation") == "VOXEL":
        edge = torch.tensor(np.asarray(params.voxel_size), device=x.device)
        dims = [int(math.ceil(s / v)) for s, v in zip(params.space_size, params.voxel_size)]
        ranges = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
    else:
        edge = h * (1 + 1e-9)
        dims = [max(1, int(s / edge) + 1) for s in params.space_size]
        ranges = [(0, b, c) for c in (-1, 0, 1) for b in (-1, 0, 1)]
    for a, i, j in _candidates(x, edge, dims, ranges, len(ranges) == 9):
        near = ((x[i] - x[j]) ** 2).sum(1) <= h * h
        i, j = i[near], j[near]
        if len(ranges) == 27:
            count = torch.bincount(i - a, minlength=1)
            rank = torch.arange(i.numel(), device=x.device) - (count.cumsum(0) - count)[i - a]
            i, j = i[rank < 32], j[rank < 32]
        out_i.append(i)
        out_j.append(j)
    i, j = torch.cat(out_i), torch.cat(out_j)
    return i, j


def _step(x, v, mu, case, consts, params, collide):
    m, h, h2 = consts.mass, consts.h, consts.h ** 2
    i, j = _pairs(x.detach(), case, consts, params)
    voxel = case.get("formulation") == "VOXEL"
    grad_c, lap_c = -45.0 / (math.pi * h ** 6), 45.0 / (math.pi * h ** 6)
    w_c = m * 315.0 / (64.0 * math.pi * h ** 9)
    n, self_pair = x.shape[0], i == j
    i, j = i[~self_pair], j[~self_pair]
    d = x[i] - x[j]
    r2 = (d * d).sum(1)
    rho = torch.zeros(n, dtype=x.dtype, device=x.device).index_add(0, i, w_c * (h2 - r2) ** 3)
    if not voxel:
        rho = rho + w_c * h2 ** 3
    p, r = consts.k * (rho - consts.rho0), r2.sqrt()
    zero = torch.zeros_like(x)
    if voxel:
        f = p / rho ** 2
        press = zero.index_add(0, i, ((f[i] + f[j]) * grad_c * (h - r) ** 2 / r)[:, None] * d)
        visc = zero.index_add(0, i, ((lap_c * (h - r) * m * mu) / (rho[i] * rho[j]))[:, None] * (v[j] - v[i]))
        visc = visc.clamp(max=1.0)
    else:
        press = zero.index_add(0, i, (m * (p[i] + p[j]) / (2 * rho[j]) * grad_c * (h - r) ** 2 / r)[:, None] * d)
        visc = zero.index_add(0, i, (m * mu / rho[j] * lap_c * (h - r))[:, None] * (v[j] - v[i]))
    ext = torch.tensor(np.asarray(params.external_force, dtype=np.float64), device=x.device)
    dt = 1.0 / params.fps
    v = v + (ext - press + visc) / rho[:, None] * dt
    x = x + v * dt
    x, v = collide(x, v)
    return x, v, rho


def _box_walls(consts, params):
    size = [float(s) for s in params.space_size]

    def collide(x, v):
        s = torch.tensor(size, dtype=x.dtype, device=x.device)
        lo, hi = x < 0, x > s
        x = torch.where(lo, torch.full_like(x, 1e-3), torch.where(hi, (s - 1e-3).expand_as(x), x))
        return x, torch.where(lo | hi, -consts.damp * v, v)

    return collide


def _streams(n, seed):
    """xoroshiro128+ state of each particle: SplitMix64 of the seed in both words, each next
    stream 2^64 draws further on."""
    mask = (1 << 64) - 1
    z = (seed + 0x9E3779B97F4A7C15) & mask
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
    s0 = s1 = z ^ (z >> 31)
    jump = 0xBEAC0467EBA5FACB | 0xD86B048B86AA9922 << 64
    out = []
    for _ in range(n):
        out.append([s0, s1])
        a = b = 0
        for bit in range(128):
            if jump >> bit & 1:
                a ^= s0
                b ^= s1
            s0, s1 = _next_state(s0, s1)
        s0, s1 = a, b
    return out


def _next_state(s0, s1):
    mask = (1 << 64) - 1
    s1 ^= s0
    return (((s0 << 55 | s0 >> 9) & mask) ^ s1 ^ (s1 << 14 & mask), (s1 << 36 | s1 >> 28) & mask)


def _pipe_walls(params, n, seed=16435234):
    """Mirror at the inlet, a random point of the inlet's disc past the outlet, reflection at
    the wall with the overshoot taken back along the velocity."""
    table = params.pipe.to_numpy()
    kept = []

    def collide(x, v):
        t = torch.tensor(table, dtype=x.dtype, device=x.device)
        xs, r = t[:, 0].contiguous(), t[:, 3]
        last = len(table) - 2
        back = x[:, 0] < 0
        x, v = x.clone(), v.clone()
        x[:, 0], v[:, 0] = torch.where(back, -x[:, 0], x[:, 0]), torch.where(back, -v[:, 0], v[:, 0])
        gone = (x[:, 0] >= xs[-1]) & ~back
        for q in gone.nonzero().flatten().tolist():
            if not kept:
                kept.extend(_streams(n, seed))
            u = []
            for _ in range(2):
                a, b = kept[q]
                u.append((((a + b) & ((1 << 64) - 1)) >> 11) * 2.0 ** -53)
                kept[q] = list(_next_state(a, b))
            rad, th = float(r[0]) * math.sqrt(u[0]), u[1] * 2.0 * math.pi
            x[q] = torch.tensor([0.0, table[0][1] + rad * math.cos(th), table[0][2] + rad * math.sin(th)])
        seg = (torch.searchsorted(xs, x[:, 0].contiguous(), right=True) - 1).clamp(0, last)
        seg = torch.where(back, 0, seg)
        r0, r1, length, base = r[seg], r[seg + 1], t[seg, 4], t[seg]
        yn, zn = x[:, 1] - base[:, 1], x[:, 2] - base[:, 2]
        hyp = (yn * yn + zn * zn).sqrt()
        out = (hyp > r0 + (r1 - r0) * (x[:, 0] - xs[seg]) / length) & ~gone
        hyp = torch.where(out, hyp, 1.0)
        ry, rz = yn / hyp, zn / hyp
        first = torch.stack([xs[seg], ry * r0, rz * r0], 1)
        edge = torch.stack([xs[seg + 1], ry * r1, rz * r1], 1) - first
        first = first + torch.stack([torch.zeros_like(yn), base[:, 1], base[:, 2]], 1)
        speed, el = v.norm(dim=1), edge.norm(dim=1)
        dist = torch.linalg.cross(edge, first - x).norm(dim=1) / el
        sin_a = torch.linalg.cross(v, edge).norm(dim=1) / (speed * el)
        hit = x - v * (dist / (sin_a + 0.001) / speed)[:, None]
        along = 2 * edge * ((edge * v).sum(1) / el ** 2)[:, None] - v
        flat = torch.stack([v[:, 0], -v[:, 1], -v[:, 2]], 1)
        new_v = torch.where((r0 == r1)[:, None], flat, along)
        new_x = hit + new_v * ((x - hit).norm(dim=1) / new_v.norm(dim=1))[:, None]
        return torch.where(out[:, None], new_x, x), torch.where(out[:, None], new_v, v)

    return collide


def _as_fp32_inputs(state, dev):
    return [torch.from_numpy(np.asarray(a)).to(dev).float().double() for a in (state.position, state.velocity)]


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind == "batch":
        parts = []
        for w in _batch_instances(case, seed):
            x, v = _as_fp32_inputs(w.state, dev)
            walls = _box_walls(w.constants, w.params)
            for _ in range(case["steps"]):
                x, v, rho = _step(x, v, w.constants.visc, case, w.constants, w.params, walls)
            parts.append(torch.cat([x.t(), v.t(), rho[None]]))
        return list(torch.cat(parts, 1))
    params, consts, state, mode = _workload(case, seed)
    x, v = _as_fp32_inputs(state, dev)
    walls = _pipe_walls(params, x.shape[0]) if mode == "PIPE" else _box_walls(consts, params)
    if kind == "gradients":
        target = _target(case, seed, x.float()).double()
        x0, v0 = x.requires_grad_(), v.requires_grad_()
        mu = torch.tensor(consts.visc, dtype=torch.float64, device=dev, requires_grad=True)
        x, v = x0, v0
        for _ in range(case["steps"]):
            x, v, _ = _step(x, v, mu, case, consts, params, walls)
        loss = ((x - target) ** 2).sum(1).mean()
        gx, gv, gmu = torch.autograd.grad(loss, (x0, v0, mu))
        return [x.detach(), v.detach(), gx, gv, gmu]
    record = []
    for _ in range(case["steps"]):
        x, v, rho = _step(x, v, consts.visc, case, consts, params, walls)
        record.append([x, v, rho])
    if kind == "frames":
        return record
    return [*x.t(), *v.t(), rho]
