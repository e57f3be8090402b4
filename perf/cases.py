"""The work that a program using this framework has it do, as cases to time.

Every case goes through the package's public entry points:

  dam    a PCISPH dam break: upload, some time steps, the state read back
         (Simulation.upload / step / state)
  sph    the same with WCSPH or original SPH
  rigid  the rigid-fluid coupling step, bodies read back too
  batch  many uneven dam breaks stepped together (Batch)
  grad   the differentiable rollout, forward and backward (adjoint.Rollout)
  fill   an OBJ-like triangle mesh filled with particles (mesh_fill)
  sort   the stable key sort on caller-owned device memory
         (upf_radix_sort_noalloc)

Sizes run from the tests' 12^3 block to the benchmark's 1M dam break.
"""
import ctypes as C
import math

import numpy as np
import torch
import torch.utils.checkpoint

import unifiedparticleframeworkcuda_amd as upf
from unifiedparticleframeworkcuda_amd import adjoint

METHODS = {"pcisph": upf.UPF_PCISPH_STATIC, "wcsph": upf.UPF_WCSPH_STATIC, "sph": upf.UPF_SPH_STATIC}
SPH_DT = 0.000253  # 0.4 h / c of the stiffness 1000 fluid


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest scene the tests step: latency and launches
        dict(name="dam_small", kind="dam", nx=12, ny=12, nz=12, steps=20, walls="thin"),
        # 65,536 particles in the corner of a box: a desktop-sized simulation
        dict(name="dam_65k", kind="dam", nx=64, ny=32, nz=32, steps=20, walls="thin"),
        # odd extents, walls sampled at half spacing with Akinci volumes
        dict(name="dam_dense_walls", kind="dam", nx=61, ny=29, nz=47, steps=20, walls="dense"),
        # the headline workload: one million fluid particles
        dict(name="dam_1m", kind="dam", nx=128, ny=64, nz=128, steps=50, walls="thin"),
        # weakly compressible SPH on the same million particles
        dict(name="wcsph_1m", kind="sph", nx=128, ny=64, nz=128, steps=50, method="wcsph"),
        # original SPH, small and ragged
        dict(name="sph_ragged", kind="sph", nx=33, ny=17, nz=25, steps=40, method="sph"),
        # rigid bodies dropped onto half a million fluid particles
        dict(name="rigid_524k", kind="rigid", nx=64, ny=128, nz=64, bodies=64, steps=10),
        # uneven independent scenes in shared launches, the step a graph replay
        dict(name="batch_96", kind="batch", scenes=96, lo=2048, hi=65536, steps=10),
        # gradient of a rollout, the gradient workload and a small one
        dict(name="grad_65k", kind="grad", nx=64, ny=32, nz=32, steps=64, iterations=5, every=8),
        dict(name="grad_small", kind="grad", nx=15, ny=11, nz=13, steps=24, iterations=3, every=6),
        # a model of 6,400 triangles turned into particles
        dict(name="fill_6400", kind="fill", nu=80, nv=41, mesh=3, scale=2.5, spacing=0.005),
        # a million z-index keys sorted on the device
        dict(name="sort_1m", kind="sort", n=1 << 20),
    ]


def draw(rng):
    def block(lo, hi, most=1 << 20):
        """A fluid lattice of about lo .. hi particles, odd extents among them."""
        n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        ax, ay = rng.uniform(0.6, 2.0), rng.uniform(0.5, 1.2)
        nz = (n / (ax * ay)) ** (1.0 / 3.0)
        e = [max(6, int(round(nz * f))) for f in (ax, ay, 1.0)]
        while e[0] * e[1] * e[2] > most:
            e[e.index(max(e))] -= 1
        return dict(nx=e[0], ny=e[1], nz=e[2])

    kind = rng.choice(["dam", "dam", "dam", "sph", "sph", "rigid", "batch", "grad", "grad", "fill", "sort"])
    if kind == "dam":
        return dict(kind=kind, **block(1500, 700000), steps=rng.randint(10, 50),
                    walls=rng.choice(["thin", "thin", "dense", "weight"]))
    if kind == "sph":
        return dict(kind=kind, **block(2000, 1 << 20), steps=rng.randint(10, 50),
                    method=rng.choice(["wcsph", "sph"]))
    if kind == "rigid":
        return dict(kind=kind, **block(30000, 500000), bodies=rng.randint(4, 64), steps=rng.randint(4, 12))
    if kind == "batch":
        lo = rng.randint(1000, 4000)
        return dict(kind=kind, scenes=rng.randint(3, 96), lo=lo, hi=lo * rng.randint(2, 16), steps=rng.randint(4, 12))
    if kind == "grad":
        return dict(kind=kind, **block(1500, 65536, 65536), steps=rng.randint(8, 64), iterations=rng.randint(2, 5),
                    every=rng.randint(4, 10))
    if kind == "fill":
        return dict(kind=kind, nu=rng.randint(16, 80), nv=rng.randint(9, 41), mesh=rng.randint(0, 999), scale=round(rng.uniform(1.0, 2.5), 3),
                    spacing=round(rng.uniform(0.005, 0.012), 4))
    return dict(kind=kind, n=int(math.exp(rng.uniform(math.log(3000), math.log(1 << 20)))))


# ------------------------------------------------------------------ the inputs
def _scene(case, seed):
    """(params, positions, types) of a dam-break case."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    sph = case["kind"] == "sph"
    walls = case.get("walls", "thin")
    if walls == "dense":
        p = upf.make_params(0.01, 0.001)
        pos, typ, _ = upf.dam_break(p, nx, ny, nz, (0.02 * nx, 0.01 * ny, 0.01 * nz), wall_rel=0.5, seed=seed)
        p.boundary_pressure_mode = upf.UPF_BOUNDARY_AKINCI
        upf.density_error_factor(p)
        return p, pos, typ
    p, pos, typ, _ = upf.standard_dam_break(nx, ny, nz, dt=SPH_DT if sph else 0.001, seed=seed)
    if sph:
        p.gas_const_wcsph = 1000.0
    if walls == "weight":  # the walls enter through the wall weight function only
        f = typ == upf.UPF_LIQUID
        pos, typ = pos[f], typ[f]
        p.add_wall_weight = 1
    return p, pos, typ


def _gradient_inputs(case, seed):
    """Scene, initial velocities and dL/dx of the mean squared distance to a
    target cloud at the initial positions (the gradient workload's loss)."""
    p, pos, typ, vel, target, f = adjoint.differentiable_dam_break(case["nx"], case["ny"], case["nz"],
                                                                   seed_v=4 + seed, seed_target=5 + seed)
    g = np.zeros((len(typ), 3), np.float32)
    g[f] = 2.0 * (pos[f, :3] - target[f]) / f.sum()
    return p, pos, typ, vel, g


def _velocities(typ, seed):
    """Initial fluid velocities, N(0, 0.1) per component."""
    v = np.zeros((len(typ), 4), np.float32)
    f = typ == upf.UPF_LIQUID
    v[f, :3] = np.random.RandomState(seed % (1 << 31)).normal(0.0, 0.1, (int(f.sum()), 3))
    return v


def _mesh(case, seed):
    """Triangles of a closed bumpy blob of radius 0.08 ((n, 3, 3) float32), the
    faces in a seeded order, and the offset that the model is placed at."""
    nu, nv = case["nu"], case["nv"]
    rng = np.random.RandomState(case["mesh"])
    k, ph = rng.uniform(1.0, 3.0, 3), rng.uniform(0.0, 2 * np.pi, 3)
    t = 2 * np.pi * np.arange(nu)[:, None] / nu
    a = np.pi * np.arange(nv)[None, :] / (nv - 1)
    r = 0.08 * (1.0 + 0.25 * np.sin(k[0] * t + ph[0]) * np.sin(k[1] * a + ph[1]) * np.cos(k[2] * (t + a) + ph[2]))
    v = np.stack([r * np.sin(a) * np.cos(t) - 0.05, r * np.cos(a) + 0.1, r * np.sin(a) * np.sin(t) + 0.04], -1)
    i, j = np.meshgrid(np.arange(nu), np.arange(nv - 1), indexing="ij")
    i1 = (i + 1) % nu
    q = np.stack([np.stack([v[i, j], v[i1, j], v[i1, j + 1]], 2), np.stack([v[i, j], v[i1, j + 1], v[i, j + 1]], 2)], 2)
    q = q.reshape(-1, 3, 3).astype(np.float32)
    rng = np.random.RandomState(seed % (1 << 31))
    return q[rng.permutation(len(q))], rng.uniform(0.0, 1.0, 3).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("dam", "sph"):
        p, pos, typ = _scene(case, seed)
        s.update(sim=upf.Simulation(p, len(typ)), pos=pos, typ=typ, method=METHODS[case.get("method", "pcisph")])
    elif kind == "rigid":
        p, pos, typ, bid, rel, bodies, _ = upf.standard_rigid_scene(case["nx"], case["ny"], case["nz"],
                                                                    n_bodies=case["bodies"])
        s.update(sim=upf.Simulation(p, len(typ)), pos=pos, typ=typ, vel=_velocities(typ, seed), bid=bid, rel=rel,
                 bodies=bodies)
    elif kind == "batch":
        sc = upf.batch_dam_breaks(case["scenes"], count_range=(case["lo"], case["hi"]))
        typ = np.concatenate([c[2] for c in sc])
        s.update(batch=upf.Batch([c[0] for c in sc], [len(c[2]) for c in sc]),
                 pos=np.concatenate([c[1] for c in sc]), typ=typ, vel=_velocities(typ, seed))
    elif kind == "grad":
        p, pos, typ, vel, g = _gradient_inputs(case, seed % (1 << 30))
        s.update(rollout=adjoint.Rollout(p, pos, typ, case["steps"], case["iterations"], case["every"]), vel=vel, g=g)
    elif kind == "fill":
        faces, offset = _mesh(case, seed)
        s.update(faces=faces, offset=offset)
    else:
        n = case["n"]
        e = max(6, int(round(n ** (1.0 / 3.0))))
        p, pos, typ, _ = upf.standard_dam_break(e, e, e, seed=seed)
        keys = np.resize(upf.device_keys(p, pos), n)
        keys = keys[np.random.RandomState(seed % (1 << 31)).permutation(n)]
        fn = upf.lib().upf_radix_sort_noalloc
        fn.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
        s.update(fn=fn, keys=torch.from_numpy(keys.view(np.int32)).cuda(),
                 out=torch.empty(n, dtype=torch.int32, device="cuda"),
                 perm=torch.empty(n, dtype=torch.int32, device="cuda"))
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("dam", "sph"):
        s["sim"].upload(s["pos"], s["typ"])
        s["sim"].step(case["steps"], s["method"])
        return s["sim"].state()
    if kind == "rigid":
        sim = s["sim"]
        sim.upload(s["pos"], s["typ"], s["vel"])
        sim.upload_bodies(s["bodies"], s["bid"], s["rel"])
        sim.step(case["steps"], upf.UPF_PCISPH_RIGID)
        out = sim.state()
        b = sim.bodies(len(s["bodies"]))
        out["bodies"] = np.array([list(x.pos) + list(x.vel) + list(x.angular_momentum) + list(x.quaternion)
                                  for x in b], np.float32)
        return out
    if kind == "batch":
        s["batch"].upload(s["pos"], s["typ"], s["vel"])
        s["batch"].step(case["steps"])
        return s["batch"].state()
    if kind == "grad":
        x, v = s["rollout"].forward(s["vel"])
        gx, gv = s["rollout"].backward(s["g"])
        return dict(x=x, v=v, gx=gx, gv=gv)
    if kind == "fill":
        return upf.mesh_fill(s["faces"], case["scale"], case["spacing"]) + s["offset"]  # as model_particles
    rc = s["fn"](case["n"], s["keys"].data_ptr(), s["out"].data_ptr(), s["perm"].data_ptr(),
                 torch.cuda.current_stream().cuda_stream)
    if rc:
        raise RuntimeError("upf_radix_sort_noalloc: %d" % rc)
    return dict(keys=s["out"], perm=s["perm"])


# ------------------------------------------------------------------ the work
def work(case):
    """Each step reads and writes positions and velocities once; per neighbour
    pair (about 30 a particle) 25 operations a pass."""
    kind = case["kind"]
    if kind == "sort":
        return dict(bytes=12.0 * case["n"], flops=0.0)
    if kind == "fill":
        nf = 2 * case["nu"] * (case["nv"] - 1)
        pts = 0.19 * 0.19 * 0.19 * (case["scale"] / case["spacing"]) ** 3
        # a point inside the mesh: the faces met along one line of a lattice column
        return dict(bytes=36.0 * nf + 12.0 * pts, flops=50.0 * pts)
    if kind == "batch":
        n = case["scenes"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
    else:
        n = case["nx"] * case["ny"] * case["nz"]
    passes = {"dam": 7, "sph": 2, "rigid": 7, "batch": 7}.get(kind, 0)
    if kind == "grad":
        passes = 3 * (1 + 2 * case["iterations"])
    return dict(bytes=64.0 * n * case["steps"] + 100.0 * n, flops=25.0 * 30 * passes * n * case["steps"])


# ------------------------------------------------------------------ 64 bits
def exact(case, seed):
    """run()'s outputs in 64 bits from plain torch.  None where it would take
    too long (long runs of many particles, the coupling step)."""
    kind = case["kind"]
    if kind == "fill":
        faces, offset = _mesh(case, seed)
        return _fill64(faces, case["scale"], case["spacing"]) + torch.tensor(offset, dtype=torch.float64)
    if kind == "grad":
        return _rollout64(case, *_gradient_inputs(case, seed % (1 << 30)))
    if kind in ("dam", "sph") and case["nx"] * case["ny"] * case["nz"] * case["steps"] <= 4000000:
        return _simulate64(case, *_scene(case, seed))
    return None


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _pairs(x, h, owner):
    """(i, j) of all pairs closer than h, i != j, i among the owners, sorted by i."""
    c = torch.floor(x / h).long()
    c = c - c.amin(0) + 1
    d = (c.amax(0) + 2).tolist()
    cell = (c[:, 0] * d[1] + c[:, 1]) * d[2] + c[:, 2]
    order = torch.argsort(cell)
    sc = cell[order]
    own = torch.nonzero(owner).flatten()
    ii, jj = [], []
    for a in (-1, 0, 1):
        for b in (-1, 0, 1):
            for e in (-1, 0, 1):
                q = cell[own] + (a * d[1] + b) * d[2] + e
                lo, hi = torch.searchsorted(sc, q), torch.searchsorted(sc, q, right=True)
                n = hi - lo
                i = torch.repeat_interleave(own, n)
                k = torch.arange(i.numel(), device=x.device) - torch.repeat_interleave(torch.cumsum(n, 0) - n, n)
                j = order[torch.repeat_interleave(lo, n) + k]
                keep = ((x[i] - x[j]).square().sum(1) < h * h) & (i != j)
                ii.append(i[keep])
                jj.append(j[keep])
    return torch.cat(ii), torch.cat(jj)


def _w(r, h):
    """KernelM4."""
    s = r / h
    t = 1.0 - s
    a = 8.0 / (math.pi * h ** 3)
    return torch.where(r < h, a * torch.where(s < 0.5, 1.0 - 6.0 * s * s + 6.0 * s ** 3, 2.0 * t ** 3), 0.0 * r)


def _simulate64(case, p, pos, typ):
    """The PCISPH, WCSPH and SPH steps of a static scene with the kernels as
    300-entry tables holding each bin's value at its start."""
    dev, f64 = _device(), torch.float64
    n, h, m, rho0, dt = len(typ), p.support_radius, p.initial_mass, p.rest_density, p.dt
    x = torch.tensor(pos[:, :3], dtype=f64, device=dev)
    v = torch.zeros_like(x)
    liq = torch.tensor(typ == upf.UPF_LIQUID, device=dev)
    lo = torch.tensor(list(p.collision_min), dtype=f64, device=dev)
    hi = torch.tensor(list(p.collision_max), dtype=f64, device=dev)
    r = h * torch.arange(300, dtype=f64, device=dev) / 300
    zero = torch.zeros(1, dtype=f64, device=dev)
    c6 = 45.0 / (math.pi * h ** 6)
    wt = torch.cat([_w(r, h), zero])
    gt = torch.cat([torch.where(r > 0, -c6 / torch.where(r > 0, r, 1.0) * (h - r) ** 2, 0.0), zero])
    lt = torch.cat([c6 * (h - r), zero])

    def bins(d):
        return (d / h * 300.0).long().clamp(max=300)

    def total(i, t):
        return torch.zeros((n,) + t.shape[1:], dtype=f64, device=dev).index_add_(0, i, t)

    akinci = p.boundary_pressure_mode == upf.UPF_BOUNDARY_AKINCI
    psi = torch.full((n,), m / rho0, dtype=f64, device=dev)
    pressure = torch.zeros(n, dtype=f64, device=dev)
    rho = torch.full((n,), rho0, dtype=f64, device=dev)
    force = torch.zeros_like(x)
    if case["kind"] == "dam" and not bool(liq.all()):
        bi, bj = _pairs(x, h, ~liq)
        k = ~liq[bj]
        s = total(bi[k], wt[bins((x[bi[k]] - x[bj[k]]).norm(dim=1))])
        psi = torch.where(liq, psi, 0.7 / (s + wt[0]) if akinci else 1.0 / s)
    down = torch.zeros_like(x)
    down[:, 1] = m * p.gravity

    def wall(y):
        """The wall weight function of the distance to the nearest face."""
        cl = torch.tensor(list(p.container_min), dtype=f64, device=dev)
        ch = torch.tensor(list(p.container_max), dtype=f64, device=dev)
        d = torch.minimum((y - cl).clamp(min=0).amin(1), (ch - y).clamp(min=0).amin(1))
        d1 = d + p.particle_radius
        d2, s1, s2 = d1 + p.spacing, p.spacing ** 2, (2 * p.spacing) ** 2
        k = wt[bins(d1)] + wt[bins(d2)]
        for q in (d1, d2):
            k = k + 2.0 * (wt[bins((q * q + s1).sqrt())] + wt[bins((q * q + s2).sqrt())])
        return torch.where(d < h - p.particle_radius, m * k, 0.0)

    for _ in range(case["steps"]):
        i, j = _pairs(x, h, liq)
        d = x[i] - x[j]
        b = bins(d.norm(dim=1))
        fj = liq[j]
        if case["kind"] == "sph":
            rho = torch.where(liq, p.kernel_self * m + total(i, wt[b] * m), 0.0)
            if p.add_wall_weight:
                rho = rho + torch.where(liq, wall(x), 0.0)
            if case["method"] == "wcsph":
                pressure = rho0 * p.gas_const_wcsph / 7.0 * ((rho / rho0) ** 7 - 1.0)
            else:
                pressure = rho0 * p.gas_const_sph * (rho / rho0 - 1.0)
            pressure = torch.where(liq, pressure.clamp(min=0.0), 0.0)
            i, j, d, b = i[fj], j[fj], d[fj], b[fj]
            g = (pressure[i] / rho[i] ** 2 + pressure[j] / rho[j] ** 2) * m * m * gt[b]
            vis = m / rho[i] * m / rho[j] * p.visc_const * lt[b]
            force = -total(i, d * g[:, None] + (v[i] - v[j]) * vis[:, None]) - down
        else:
            t = (v[i] - v[j]) * (torch.where(fj, (m / rho0) ** 2 * p.visc_const * lt[b], 0.0))[:, None]
            if akinci:
                q = pressure[i] / rho[i] ** 2 * m * rho0 * psi[j] * gt[b]
                t = t + d * torch.where(fj, 0.0, q)[:, None]
            ext = -total(i, t) - down
            fp = torch.zeros_like(x)
            pressure = torch.zeros_like(pressure)
            mj = torch.where(fj, m, rho0 * psi[j]) if akinci else torch.full_like(psi[j], m)
            too_large, it = True, 0
            while it < p.min_loops or (too_large and it < p.max_loops):
                xs = torch.minimum(torch.maximum(x + (v + (ext + fp) * (dt / m)) * dt, lo), hi)
                xs = torch.where(liq[:, None], xs, x)
                dist = (xs[i] - xs[j]).norm(dim=1)
                now = p.kernel_self * m + total(i, torch.where(dist < h, wt[bins(dist)] * mj, 0.0))
                if p.add_wall_weight:
                    now = now + wall(xs)
                rho = torch.where(liq, now, rho)
                pressure = torch.where(liq, pressure + ((now - rho0).clamp(min=0) * p.density_error_factor).clamp(min=0),
                                       0.0)
                g = (pressure[i] + torch.where(fj, pressure[j], 0.0)) / rho0 ** 2 * m * mj * gt[b]
                fp = -total(i, d * g[:, None])
                it += 1
                if max(0.1 * float(now[liq].max()) - 100.0, 0.0) < p.max_density_error_allowed:
                    too_large = False
            force = ext + fp
        force = torch.where(liq[:, None], force, 0.0)
        v = torch.where(liq[:, None], v + force / m * dt, v)
        x = torch.where(liq[:, None], x + v * dt, x)
        out = ((x < lo) | (x > hi)) & liq[:, None]
        v = torch.where(out, -0.5 * v, v)
        x = torch.where(out, torch.minimum(torch.maximum(x, lo), hi), x)

    def four(t):
        return torch.cat([t, torch.zeros_like(t[:, :1])], 1).cpu()

    # A distance within rounding of a table bin's edge falls into either bin, so
    # the velocities, pressures and forces of single particles of a 32-bit and a
    # 64-bit run part within a few steps; positions and densities stay close.
    return dict(pos=four(x), vel=None, rho=rho.cpu(), p=None, force=None, psi=psi.cpu(), type=torch.tensor(typ))

def _rollout64(case, p, pos, typ, vel, g):
    """The differentiable rollout and its gradient by automatic differentiation."""
    dev, f64 = _device(), torch.float64
    h, m, rho0, dt = p.support_radius, p.initial_mass, p.rest_density, p.dt
    fluid = torch.tensor(typ == upf.UPF_LIQUID, device=dev)
    n = len(typ)
    lo = torch.tensor(list(p.collision_min), dtype=f64, device=dev)
    hi = torch.tensor(list(p.collision_max), dtype=f64, device=dev)
    c6 = 45.0 / (math.pi * h ** 6)
    fd, kb = p.force_distance, 2.0 * p.max_boundary_force / p.force_distance
    down = torch.zeros((n, 3), dtype=f64, device=dev)
    down[:, 1] = m * p.gravity

    def total(i, t):
        return torch.zeros((n,) + t.shape[1:], dtype=f64, device=dev).index_add(0, i, t)

    def clamp(y):
        return torch.minimum(torch.maximum(y, lo), hi)

    def step(x, v):
        with torch.no_grad():
            i, j = _pairs(x, h, fluid)
            fj = fluid[j]
        d = x[i] - x[j]
        r = d.square().sum(1).sqrt()
        s = torch.where(fj, (m / rho0) ** 2 * p.visc_const * c6 * (h - r), 0.0)
        ext = -total(i, (v[i] - v[j]) * s[:, None]) - down
        ext = ext + (lo + fd - x).clamp(min=0) * kb - (x + fd - hi).clamp(min=0) * kb
        gk = -c6 * (h - r) ** 2 / r
        fp, pr = torch.zeros_like(x), torch.zeros(n, dtype=f64, device=dev)
        for _ in range(case["iterations"]):
            xs = torch.where(fluid[:, None], clamp(x + (v + (ext + fp) * (dt / m)) * dt), x)
            rs = (xs[i] - xs[j]).square().sum(1).sqrt()
            rho = m * 8.0 / (math.pi * h ** 3) + total(i, m * _w(rs, h))
            pr = torch.where(fluid, pr + p.density_error_factor * torch.nn.functional.softplus(rho - rho0, threshold=40),
                             0.0)
            fp = -total(i, d * (gk * (pr[i] + pr[j]) * m * m / rho0 ** 2)[:, None])
        v2 = v + (ext + fp) * (dt / m)
        return torch.where(fluid[:, None], clamp(x + v2 * dt), x), torch.where(fluid[:, None], v2, v)

    x0 = torch.tensor(pos[:, :3], dtype=f64, device=dev, requires_grad=True)
    v0 = torch.tensor(vel, dtype=f64, device=dev, requires_grad=True)
    x, v = x0, v0
    for _ in range(case["steps"]):
        x, v = torch.utils.checkpoint.checkpoint(step, x, v, use_reentrant=False)
    gx, gv = torch.autograd.grad(x, (x0, v0), torch.tensor(g, dtype=f64, device=dev))
    keep = fluid[:, None]
    return dict(x=x.detach().cpu(), v=v.detach().cpu(), gx=torch.where(keep, gx, 0.0).cpu(),
                gv=torch.where(keep, gv, 0.0).cpu())


def _fill64(faces, scale, spacing):
    """Lattice points that the segment from outside the model's box reaches
    through an odd number of faces."""
    dev, f64 = _device(), torch.float64
    t = torch.tensor(faces, dtype=f64, device=dev)
    mn, mx = t.reshape(-1, 3).amin(0).clamp(max=0), t.reshape(-1, 3).amax(0).clamp(min=0)
    n = [int(math.floor(float(e) * scale / spacing)) + 1 for e in mx - mn]
    ix = torch.arange(n[0], dtype=f64, device=dev)[:, None, None]
    half = 0.5 * (torch.arange(n[0], device=dev) % 2).to(f64)[:, None, None]
    iy = torch.arange(n[1], dtype=f64, device=dev)[None, :, None] + half
    iz = torch.arange(n[2], dtype=f64, device=dev)[None, None, :] + half
    pts = torch.stack(torch.broadcast_tensors(ix, iy, iz), -1).reshape(-1, 3) * (spacing / scale) + mn
    o = mn - spacing
    e1, e2 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    a = o - t[:, 0]
    inside = torch.zeros(len(pts), dtype=torch.bool, device=dev)
    chunk = max(1, (1 << 28) // max(1, len(t)))
    for k in range(0, len(pts), chunk):
        d = pts[k:k + chunk] - o
        # the segment parameter and the barycentric coordinates, scaled by den
        den = -(d @ nrm.T)
        sg = torch.sign(den)
        tt = (a * nrm).sum(1)[None] * sg
        u = (d @ torch.linalg.cross(e2, a).T) * sg
        w = (d @ torch.linalg.cross(a, e1).T) * sg
        ad = den.abs()
        hit = (ad > 0) & (tt >= 0) & (tt <= ad) & (u >= 0) & (w >= 0) & (u + w <= ad)
        inside[k:k + chunk] = (hit.sum(1) % 2) == 1
    return ((pts[inside] - mn) * scale).cpu()
