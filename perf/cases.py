"""The work a user of this framework has it do, as cases that can be timed.

Every case is a Position Based Fluids scene: jittered lattice blocks at
spacing 0.05 (h = 0.1) dropped in a box, with the physics of the benchmark
workloads.  `kind` names the public entry point a program calls:

  call      hip.hip_step(params, state): the stateless drop-in for the
            reference's cuda_step, host arrays in and out, one substep
  inplace   hip.step_noalloc on device arrays, for programs that may not
            allocate: the fixed per-GPU scratch array
  resident  HipSolver: upload, the substeps of one output frame (30 frames/s
            at 120 substeps/s is 4), download; `graph` replays a captured
            substep
  batch     HipSolver over a ragged ensemble of independent scenes
  grad      HipSolver.forward_record + backward: the gradient of a rollout,
            as an inverse problem takes it in every iteration

`warm` substeps have run before the pass: 0 is the lattice just released;
after some tens of substeps the block has hit the walls, particles pile up
on them and spray is in the air, so the same size is other work.
"""
import math

import numpy as np
import torch

from fluidsimulator_amd import hip
from fluidsimulator_amd.params import Params, State

SPACING = 0.05
H = 0.1
# Neighbors of a particle of the released lattice (27 inside, fewer at faces).
NEIGHBORS = 26.6


def listed():
    return [
        # one substep of a small scene through the reference's own call shape
        _case("call_1728", "call", (12, 12, 12), box=(3.0, 3.0, 3.0), flags=True, steps=1),
        # a serving loop's scene in the scratch array; odd dimensions
        _case("inplace_4199", "inplace", (19, 17, 13), box=(3.0, 3.0, 3.0), flags=True, steps=4),
        # an interactive scene, one frame, launch latency hidden by a graph
        _case("frame_2431_graph", "resident", (17, 13, 11), box=(3.0, 3.0, 3.0), flags=True,
              steps=4, warm=16, graph=True),
        # the plain dam break (240-step workload), two frames from its release
        _case("dam_32768", "resident", (32, 32, 32), box=(4.0, 3.0, 2.0), flags=False, steps=8),
        # the same block with every flag while it splashes
        _case("dam_32768_splash", "resident", (32, 32, 32), box=(4.0, 3.0, 2.0), flags=True,
              steps=4, warm=40),
        # the double dam break (262,144 particles, all flags): released, and splashing
        _case("double_262144", "resident", (64, 64, 32), blocks=2, box=(8.0, 4.0, 4.0),
              flags=True, steps=4),
        _case("double_262144_splash", "resident", (64, 64, 32), blocks=2, box=(8.0, 4.0, 4.0),
              flags=True, steps=4, warm=24),
        # the million-particle block: its first frame, and piled up on the walls
        _case("block_1048576", "resident", (128, 128, 64), box=(12.0, 8.0, 4.0), flags=True,
              steps=4),
        _case("block_1048576_piled", "resident", (128, 128, 64), box=(12.0, 8.0, 4.0),
              flags=True, steps=2, warm=30),
        # an ensemble of uneven dam breaks (2 million particles in all), under way
        _case("ensemble_256", "batch", (8, 32, 0), box=(3.0, 3.0, 3.0), flags=True, steps=2,
              warm=24, scenes=256),
        # one iteration of an inverse problem: four small scenes of the fitting
        # driver, checkpointed, and the 65,536-particle rollout
        _case("grad_fit_4x1920", "grad", (16, 12, 10), box=(4.0, 3.0, 2.0), flags=True, steps=20,
              every=10, scenes=4),
        _case("grad_65536", "grad", (64, 32, 32), box=(4.0, 3.0, 2.0), flags=True, steps=10,
              every=10),
    ]


def _case(name, kind, dims, box, flags, steps, warm=0, graph=False, blocks=1, scenes=1, every=0,
          scorr_n=4, slanted=False):
    """dims: the lattice of each block; for a batch (smallest edge, largest edge, 0)."""
    c = {"kind": kind, "nx": dims[0], "ny": dims[1], "nz": dims[2], "blocks": blocks,
         "box_x": box[0], "box_y": box[1], "box_z": box[2], "flags": flags, "steps": steps,
         "warm": warm, "graph": graph, "scenes": scenes, "every": every, "scorr_n": scorr_n,
         "slanted": slanted}
    if name:
        c["name"] = name
    return c


def draw(rng):
    kind = rng.choice(["call", "inplace", "resident", "resident", "resident", "resident", "batch",
                       "grad"])
    flags = rng.random() < 0.7
    scorr_n = rng.choice([2, 3, 4, 4])
    slanted = rng.random() < 0.25

    def block(lo, hi):
        """A lattice of about a log-uniform number of particles, no edge rule."""
        n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        e = n ** (1.0 / 3.0)
        nx = max(4, round(e * rng.uniform(0.8, 1.6)))
        ny = max(4, round(e * rng.uniform(0.7, 1.3)))
        nz = max(4, int(n / (nx * ny)))
        return nx, ny, nz

    def room(d):
        return tuple(round(SPACING * k * rng.uniform(1.3, 2.5) + 0.5, 3) for k in d)

    if kind == "call":
        d = block(500, 40000)
        return _case(None, kind, d, room(d), flags, 1, scorr_n=scorr_n, slanted=slanted)
    if kind == "inplace":
        d = block(500, 30000)
        return _case(None, kind, d, room(d), flags, rng.randint(1, 8), scorr_n=scorr_n,
                     slanted=slanted)
    if kind == "resident":
        d = block(1500, 800000)
        big = d[0] * d[1] * d[2] > 100000
        return _case(None, kind, d, room(d), flags, rng.randint(2, 4) if big else rng.randint(2, 8),
                     warm=rng.choice([0, 0, 8, 16, 28]) if flags else rng.choice([0, 4, 12]),
                     graph=rng.random() < 0.4, scorr_n=scorr_n, slanted=slanted)
    if kind == "batch":
        hi = rng.randint(10, 32)
        return _case(None, kind, (rng.randint(6, 10), hi, 0), (3.0, 3.0, 3.0), flags,
                     rng.randint(1, 3), warm=rng.choice([0, 8, 24]), scenes=rng.randint(4, 200),
                     graph=rng.random() < 0.4, scorr_n=scorr_n)
    d = block(1500, 50000)
    steps = rng.randint(3, 10)
    return _case(None, kind, d, room(d), True, steps, every=rng.choice([steps, steps, 4]),
                 scenes=rng.choice([1, 1, 2]), scorr_n=scorr_n)


def _solver_params(c):
    p = Params(dt=float(np.float32(1.0 / 120.0)), density=1000.0, particle_mass=0.125, h=H,
               particle_radius=0.025, epsilon=100.0, solver_iterations=4,
               plane_restitution=0.05, plane_friction=0.1, external_forces=(0.0, -9.8, 0.0))
    p.set_box(c["box_x"], c["box_y"], c["box_z"])
    if c["slanted"]:  # a ramp across the far lower edge of the box
        p.add_plane_normalized(-1.0, 2.0, 0.0, -0.35 * c["box_x"])
    if c["flags"]:
        p.enable_scorr, p.scorr_k, p.scorr_n, p.scorr_dq_coeff = True, 0.1, c["scorr_n"], 0.2
        p.enable_xsph, p.visc_c = True, 0.01
        p.enable_vorticity, p.vort_epsilon = True, 5e-4
    if c["kind"] == "grad":
        # the gradient of a longer rollout stays bounded with these
        p.enable_vorticity = False
        p.epsilon, p.scorr_k, p.scorr_dq_coeff, p.visc_c = 600.0, 5e-5, 0.3, 2e-4
    return p


def _lattice(rng, nx, ny, nz, ox=0.0):
    """A block of lattice sites with a tenth of a spacing of jitter, x fastest."""
    iz, iy, ix = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    pos = np.stack([ix.ravel(), iy.ravel(), iz.ravel()]) + 0.5
    pos = SPACING * (pos + 0.1 * (2.0 * rng.random(pos.shape) - 1.0))
    pos[0] += ox
    return pos.astype(np.float32)


def _scenes(c, seed):
    """Parameters, positions and velocities of each scene of a case."""
    rng = np.random.default_rng(seed)
    out = []
    if c["kind"] == "batch":
        # the sizes are the case's, the seed moves particles only
        sizes = np.random.default_rng(1000 * c["nx"] + c["ny"]).integers(
            c["nx"], c["ny"] + 1, (c["scenes"], 3))
        for nx, ny, nz in sizes:
            p = _solver_params(c)
            p.external_forces = (0.0, float(np.float32(-rng.uniform(8.0, 12.0))), 0.0)
            pos = _lattice(rng, nx, ny, nz)
            v0 = rng.uniform(-1.0, 1.0, (3, 1))
            out.append((p, pos, np.repeat(v0, pos.shape[1], 1).astype(np.float32)))
        return out
    for _ in range(c["scenes"]):
        blocks = [_lattice(rng, c["nx"], c["ny"], c["nz"],
                           0.0 if b == 0 else c["box_x"] - SPACING * c["nx"])
                  for b in range(c["blocks"])]
        pos = np.concatenate(blocks, 1)
        vel = np.zeros_like(pos)
        if c["kind"] == "grad":
            vel = (0.5 * rng.standard_normal(pos.shape)).astype(np.float32)
        out.append((_solver_params(c), pos, vel))
    return out


def _particles(c):
    if c["kind"] != "batch":
        return c["nx"] * c["ny"] * c["nz"] * c["blocks"] * c["scenes"]
    sizes = np.random.default_rng(1000 * c["nx"] + c["ny"]).integers(
        c["nx"], c["ny"] + 1, (c["scenes"], 3))
    return int(sizes.prod(1).sum())


def _loss_gradient(n, seed):
    rng = np.random.default_rng([seed, 1])
    return (rng.standard_normal((3, n)).astype(np.float32),
            rng.standard_normal((3, n)).astype(np.float32))


def prepare(c, seed):
    sc = _scenes(c, seed)
    params = [p for p, _, _ in sc]
    pos = np.concatenate([x for _, x, _ in sc], 1)
    vel = np.concatenate([v for _, _, v in sc], 1)
    state = {"case": c, "params": params[0]}
    if c["kind"] == "call":
        return dict(state, pos=pos, vel=vel)
    if c["kind"] == "inplace":
        return dict(state, pos=torch.from_numpy(pos).cuda(), vel=torch.from_numpy(vel).cuda())
    solver = hip.HipSolver(params, [x.shape[1] for _, x, _ in sc])
    if c["warm"]:
        solver.upload(pos, vel)
        solver.step(c["warm"])
        st = solver.download()
        pos, vel = st.pos, st.vel
    state.update(solver=solver, pos=pos, vel=vel)
    if c["kind"] == "grad":
        state["dpos"], state["dvel"] = _loss_gradient(pos.shape[1], seed)
    return state


def run(s):
    c = s["case"]
    if c["kind"] == "call":
        st = State(s["pos"].copy(), s["vel"].copy(), 0.0)
        for _ in range(c["steps"]):
            hip.hip_step(s["params"], st)
        return {"pos": st.pos, "vel": st.vel}
    if c["kind"] == "inplace":
        pos, vel = s["pos"].clone(), s["vel"].clone()
        hip.step_noalloc(s["params"], pos.shape[1], pos.data_ptr(), vel.data_ptr(), 0.0,
                         c["steps"], torch.cuda.current_stream().cuda_stream)
        return {"pos": pos, "vel": vel}
    solver = s["solver"]
    solver.upload(s["pos"], s["vel"])
    if c["kind"] == "grad":
        solver.forward_record(c["steps"], c["every"])
        st = solver.download()
        dx, dv, dg = solver.backward(s["dpos"], s["dvel"])
        return {"pos": st.pos, "vel": st.vel, "dpos0": dx, "dvel0": dv, "dgravity": dg}
    solver.step(c["steps"], graph=c["graph"])
    st = solver.download()
    return {"pos": st.pos, "vel": st.vel}


def work(c):
    """State in and out of every substep; the pair terms of the lattice's
    neighbors in every pass (piled-up scenes have more pairs)."""
    n, t, iters = _particles(c), c["steps"], 4
    pair = iters * (30 + 30)
    if c["flags"]:
        pair += 22 + (0 if c["kind"] == "grad" else 35 + 30)
    per_step = n * (NEIGHBORS * pair + 150)
    nbytes = 48.0 * n * (t + 1)
    if c["kind"] == "grad":
        # the reverse pass reads each iterate and its sums again and carries
        # the position and velocity adjoints; about twice the pair arithmetic
        per_step *= 3
        nbytes += n * t * (iters * 32.0 + 48.0) + 48.0 * n
    return {"bytes": nbytes, "flops": float(per_step * t)}


# ---------------------------------------------------------------- 64 bits


def _pairs(p, h2):
    """Ordered pairs (i, j), i != j, closer than h."""
    n, step, got = p.shape[0], 1024, []
    for a in range(0, n, step):
        d = p[a:a + step, None, :] - p[None, :, :]
        r2 = (d * d).sum(-1)
        k = torch.arange(a, min(n, a + step), device=p.device)
        r2[k - a, k] = 2.0 * h2
        i, j = torch.nonzero(r2 < h2, as_tuple=True)
        got.append(torch.stack([i + a, j]))
    return torch.cat(got, 1)


def _substep64(x, v, g, p, neighbors):
    """One PBF substep on float64 tensors x, v of shape (n, 3), differentiable
    with the pair list fixed.  neighbors(p0) lists the pairs."""
    f = lambda a: float(np.float32(a))  # noqa: E731  (parameters are float32)
    n, dt, h = x.shape[0], f(p.dt), f(p.h)
    h2, m, rho0 = h * h, f(p.particle_mass), f(p.density)
    c6, cs = 315.0 / (64.0 * math.pi * h ** 9), -45.0 / (math.pi * h ** 6)
    min_r2 = (f(0.01) * h) ** 2
    va = v + g * dt
    q = x + va * dt
    i, j = neighbors(q.detach())

    def total(t):
        z = torch.zeros((n,) + t.shape[1:], dtype=t.dtype, device=t.device)
        return z.index_add(0, i, t)

    def pair(a):
        d = a[i] - a[j]
        r2 = (d * d).sum(1)
        act = (r2 < h2).detach()
        r = torch.sqrt(torch.clamp(r2, min=min_r2))
        W = torch.where(act, c6 * (h2 - r2) ** 3, torch.zeros_like(r2))
        F = torch.where(act, cs * (h - r) ** 2, torch.zeros_like(r))
        return d, W, F

    dq = f(p.scorr_dq_coeff) * h
    inv_wdq = 1.0 / (c6 * (h2 - dq * dq) ** 3)
    rho = None
    for _ in range(int(p.solver_iterations)):
        d, W, F = pair(q)
        rho = m * (c6 * h2 ** 3 + total(W))
        G = F[:, None] * d
        S = total(G)
        Q = (m / rho0) ** 2 * (total((G * G).sum(1)) + (S * S).sum(1))
        lam = -(rho / rho0 - 1.0) / (Q + f(p.epsilon))
        sv = lam[i] + lam[j]
        if p.enable_scorr:
            sv = sv - f(p.scorr_k) * (W * inv_wdq) ** int(p.scorr_n)
        q = q + total((sv * F)[:, None] * d) / rho0
        for a in p.planes:
            nrm = torch.tensor(np.asarray(a[:3], np.float32).astype(np.float64), device=x.device)
            pen = f(a[3]) - q @ nrm
            q = q + torch.where((pen > 0).detach(), pen, torch.zeros_like(pen))[:, None] * nrm
    vel = (q - x) / dt
    d, W, F = pair(q)
    if p.enable_xsph:
        mu = m / rho
        vel = vel + f(p.visc_c) * total((W * mu[j])[:, None] * (vel[j] - vel[i]))
    if p.enable_vorticity:
        G = F[:, None] * d
        om = total(torch.linalg.cross(vel[j] - vel[i], G))
        w = om.norm(dim=1)
        eta = total((w[j] - w[i])[:, None] * G)
        ln = eta.norm(dim=1, keepdim=True)
        nrm = torch.where(ln > f(p.vort_norm_eps), eta / ln.clamp(min=1e-300),
                          torch.zeros_like(eta))
        vel = vel + dt * f(p.vort_epsilon) * torch.linalg.cross(nrm, om)
    for a in p.planes:
        nrm = torch.tensor(np.asarray(a[:3], np.float32).astype(np.float64), device=x.device)
        touch = ((q @ nrm - f(a[3])) <= 0).detach()[:, None]
        vn = (vel @ nrm)[:, None]
        back = torch.where(vn < 0, -f(p.plane_restitution) * vn, vn)
        vel = torch.where(touch, (vel - vn * nrm) * (1.0 - f(p.plane_friction)) + back * nrm, vel)
    return q, vel


def exact(c, seed):
    """The pass in 64 bits.  A few substeps of a released lattice can be
    followed there; later the map amplifies a rounding so much that two
    trajectories have nothing to do with each other, and a gradient of many
    particles needs too much memory."""
    n = _particles(c)
    if c["warm"] or c["kind"] == "batch" or n > 40000 or c["slanted"]:
        return None
    if c["kind"] == "grad":
        if n * c["steps"] > 160000:
            return None
    elif c["steps"] > 1:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    parts = []
    gx, gv = _loss_gradient(n, seed)
    at = 0
    for p, pos, vel in _scenes(c, seed):
        k = pos.shape[1]
        x, v = (torch.from_numpy(a.T.astype(np.float64)).to(dev) for a in (pos, vel))
        g = torch.tensor(np.asarray(p.external_forces, np.float32).astype(np.float64), device=dev)
        h2 = float(np.float32(p.h)) ** 2
        if c["kind"] != "grad":
            with torch.no_grad():
                for _ in range(c["steps"]):
                    x, v = _substep64(x, v, g, p, lambda q: _pairs(q, h2))
            parts.append((x.T, v.T))
            continue
        ins = [t.requires_grad_() for t in (x, v, g)]
        for _ in range(c["steps"]):
            x, v = _substep64(x, v, g, p, lambda q: _pairs(q, h2))
        lx, lv = (torch.from_numpy(a[:, at:at + k].T.astype(np.float64)).to(dev) for a in (gx, gv))
        grads = torch.autograd.grad((x * lx).sum() + (v * lv).sum(), ins)
        parts.append((x.detach().T, v.detach().T, grads[0].T, grads[1].T, grads[2][None]))
        at += k
    cat = [torch.cat([q[k] for q in parts], 0 if k == 4 else 1).cpu().numpy()
           for k in range(len(parts[0]))]
    return dict(zip(("pos", "vel", "dpos0", "dvel0", "dgravity"), cat))
