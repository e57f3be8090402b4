"""Seeded scenes shared by the tests (generated by the library's host code)."""
import ctypes as C

import numpy as np

import unifiedparticleframeworkcuda_amd as upf


def dam_break(n=16, seed=0, mode=upf.UPF_BOUNDARY_CPU_REF, dt=0.001):
    """Config-0 layout (lattice n^3 in a (2n, n, n)-spacing box), scaled to n."""
    p, pos, typ, nf = upf.standard_dam_break(n, n, n, dt=dt, seed=seed)
    p.boundary_pressure_mode = mode
    return p, pos, typ, nf


def config1_shape(scale=1):
    """The 1M-particle dam break: 128 x 64 x 128 lattice in a 2.56 x 0.64 x 1.28 m box (scale divides it)."""
    nx, ny, nz = 128 // scale, 64 // scale, 128 // scale
    return upf.standard_dam_break(nx, ny, nz)


def with_pile(p, pos, typ, count):
    """The scene, its particles in their order, with `count` wall particles between them that are piled into one
    cell far from the fluid."""
    width = p.block_size / np.array(list(p.scales))
    cell = np.floor((pos[typ == upf.UPF_FROZEN, :3].max(0) - 1.5 * width) / width)
    rng = np.random.RandomState(count)
    n = len(typ) + count
    mine = np.zeros(n, bool)
    mine[rng.choice(n, len(typ), replace=False)] = True
    x, t = np.zeros((n, 4), np.float32), np.full(n, upf.UPF_FROZEN, np.int32)
    x[mine], t[mine] = pos, typ
    x[~mine, :3] = (cell + 0.3 + rng.uniform(0.0, 0.3, (count, 3))) * width
    return x, t


def sparse_grid(p, edge=6.0):
    """Puts the scene of p into a virtual box of `edge` metres: a cell table far larger than the particles fill."""
    vec = C.c_float * 3
    upf.check("upf_params_set_domain", upf.lib().upf_params_set_domain(
        C.byref(p), vec(edge, edge, edge), vec(*p.collision_min), vec(*p.collision_max)))
    return p
