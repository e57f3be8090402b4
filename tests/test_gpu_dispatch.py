"""The kernels that a step takes by its size: 16, 4 or one lane per particle
over packed rows or delta-coded lists, builds with 16, 4 or one wave per window
of 64 slots, the sort by cells or by key.  Either side of every line, against
the separate list build and passes (which the size does not change) or against
the oracle, bit for bit."""
import numpy as np
import pytest

import oracle_lib as ol
import scenes
import unifiedparticleframeworkcuda_amd as upf
from unifiedparticleframeworkcuda_amd import adjoint as adj
from unifiedparticleframeworkcuda_amd import autotune

pytestmark = pytest.mark.gpu

BOTH = [upf.UPF_BOUNDARY_CPU_REF, upf.UPF_BOUNDARY_AKINCI]


def _of_size(total, mode):
    """A dam break of exactly `total` particles: the fluid cut to the number that fits beside the walls."""
    e = int(round((total / 1.35) ** (1.0 / 3.0)))
    p, pos, typ, _ = upf.standard_dam_break(e, e, e + 12, dt=0.000253)
    assert len(typ) >= total
    keep = np.ones(len(typ), bool)
    keep[np.flatnonzero(typ == upf.UPF_LIQUID)[-(len(typ) - total):]] = len(typ) == total
    p.boundary_pressure_mode = mode
    return p, np.ascontiguousarray(pos[keep]), typ[keep]


def _states(p, pos, typ, method, steps, *tunings):
    out = []
    for t in tunings:
        sim = upf.Simulation(p, len(typ))
        sim.set_tuning(dict(autotune.DEFAULT, **t))
        sim.upload(pos, typ)
        sim.step(steps, method)
        out.append(dict(sim.state(), K=sim.stats()[0]))
        sim.close()
    return out


def _equal(a, b):
    for k in a:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("total", [24575, 24576, 196607, 196608])
@pytest.mark.parametrize("method,mode", [(upf.UPF_PCISPH_STATIC, BOTH[0]), (upf.UPF_PCISPH_STATIC, BOTH[1]),
                                         (upf.UPF_SPH_STATIC, BOTH[0]), (upf.UPF_WCSPH_STATIC, BOTH[0])])
def test_fused_steps_equal_separate_kernels_around_the_lines(gpu, total, method, mode):
    p, pos, typ = _of_size(total, mode)
    print("dispatch: %d particles, method %d, mode %d" % (len(typ), method, mode), flush=True)
    assert len(typ) == total
    _equal(*_states(p, pos, typ, method, 3, dict(), dict(nbr_fuse=0)))


@pytest.mark.parametrize("method,mode", [(upf.UPF_PCISPH_STATIC, BOTH[1]), (upf.UPF_SPH_STATIC, BOTH[0])])
@pytest.mark.parametrize("total", [30011, 200003])
def test_steps_equal_the_oracle(gpu, total, method, mode):
    p, pos, typ = _of_size(total, mode)
    print("dispatch oracle: %d particles, method %d, mode %d" % (len(typ), method, mode), flush=True)
    g, = _states(p, pos, typ, method, 2, dict())
    o = ol.OracleSim(p, pos, None, typ)
    o.step(2, method)
    r = o.state(pcisph=method == upf.UPF_PCISPH_STATIC)
    f = typ == upf.UPF_LIQUID
    for k in ("pos", "vel", "force"):
        assert np.array_equal(g[k][f, :3], r[k][f, :3]), k
    for k in ("rho", "p"):
        assert np.array_equal(g[k][f], r[k][f]), k


@pytest.mark.parametrize("mode", BOTH)
def test_coupling_with_four_waves_per_window_equals_the_oracle(gpu, mode):
    p, pos, typ, bid, rel, bodies, _ = upf.standard_rigid_scene(24, 24, 32, 4, mode=mode)
    print("dispatch coupling: %d particles, mode %d" % (len(typ), mode), flush=True)
    assert 24576 <= len(typ) < 196608
    sim = upf.Simulation(p, len(typ))
    sim.upload(pos, typ)
    sim.upload_bodies(bodies, bid, rel)
    o = ol.OracleSim(p, pos, None, typ)
    o.upload_bodies(bodies, bid, rel, rel[:, 3].copy())
    sim.step(3, upf.UPF_PCISPH_RIGID)
    o.step(3, upf.UPF_PCISPH_RIGID)
    g, r = sim.state(), o.state()
    f = typ != upf.UPF_FROZEN
    assert np.array_equal(g["pos"][:, :3], r["pos"][:, :3]) and np.array_equal(g["vel"][:, :3], r["vel"][:, :3])
    assert np.array_equal(g["force"][f, :3], r["force"][f, :3])
    assert np.array_equal(sim.stats()[0], o.stats()[0])


@pytest.mark.parametrize("mode", BOTH)
@pytest.mark.parametrize("lattice_rel", [1.0025, 0.9])
def test_union_and_packed_lists_equal_delta_coded_lists(gpu, mode, lattice_rel):
    """Eight rounds per build keep the loop on the delta-coded lists at this size; four take the packed rows."""
    p = upf.make_params(0.01, 0.001)
    pos, typ, _ = upf.dam_break(p, 24, 16, 20, (0.48, 0.32, 0.4), lattice_rel=lattice_rel)
    upf.density_error_factor(p)
    p.boundary_pressure_mode = mode
    coded, union, packed = _states(p, pos, typ, upf.UPF_PCISPH_STATIC, 6, dict(nbr_rounds=8), dict(loop_list=2), dict())
    _equal(coded, union)
    _equal(coded, packed)


@pytest.mark.parametrize("use_graph", [1, 0, 2])
def test_batch_on_sparse_grids_equals_plain(gpu, use_graph):
    """Cell tables too sparse for the counting: the batch sorts by key, then by scene."""
    some = [(scenes.sparse_grid(s[0]),) + tuple(s[1:]) for s in upf.batch_dam_breaks(3, seed=5, count_range=(300, 4000))]
    assert all(s[0].grid_dim == 256 for s in some)
    print("sparse batch: counts %s" % [len(s[2]) for s in some], flush=True)
    b = upf.Batch.from_scenes(some)
    b.step(2, use_graph=use_graph)
    b.step(3, use_graph=use_graph)
    st = b.state()
    b.close()
    off = 0
    for i, (p, pos, typ) in enumerate(s[:3] for s in some):
        plain, = _states(p, pos, typ, upf.UPF_PCISPH_STATIC, 5, dict())
        if i == 0:
            o = ol.OracleSim(p, pos, None, typ)
            o.step(5, upf.UPF_PCISPH_STATIC)
            assert np.array_equal(plain["pos"][:, :3], o.state()["pos"][:, :3])
        for k in ("pos", "vel", "rho"):
            assert np.array_equal(st[k][off:off + len(typ)], plain[k]), k
        off += len(typ)


def test_rollout_on_a_sparse_grid_matches_the_oracle(gpu):
    p, pos, typ, vel, target, f = adj.differentiable_dam_break(9, 8, 7)
    scenes.sparse_grid(p)
    assert p.grid_dim == 256
    print("sparse rollout: %d particles" % len(typ), flush=True)
    r = adj.Rollout(p, pos, typ, 5, 2, checkpoint_every=2)
    x, v = r.forward(vel)
    g = (x - pos[:, :3]).astype(np.float64)
    gx, gv = r.backward(g)
    r.close()
    xo, vo, ox, ov = ol.diff_run(p, pos, vel, typ, 5, 2, gpos=g.astype(np.float32).astype(np.float64), precision=32)
    # the bounds of the dense grid's test: expf / log1pf are the only other source
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)
    assert np.abs(x - xo).max() < 2e-6
    assert np.abs(v - vo).max() < 1e-4 * max(np.abs(vo).max(), 1e-3)
    assert rel(gv, ov) < 1e-4 and rel(gx, ox) < 1e-4
