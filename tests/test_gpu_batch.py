"""Batched form: many uneven scenes stepped together must give, scene by
scene, exactly what a plain simulation of that scene gives (same kernels, same
per-scene neighbour order, per-scene loop control), with and without the
whole step replayed as a hipGraph; and the plain path equals the oracle.
"""
import ctypes as C

import numpy as np
import pytest

import unifiedparticleframeworkcuda_amd as upf
import oracle_lib as ol

pytestmark = pytest.mark.gpu


def _scenes(n_scenes=6, seed=11, mode=upf.UPF_BOUNDARY_CPU_REF):
    # uneven: 300 .. 4000 fluid particles, aspect ratios 0.5 .. 2
    sc = upf.batch_dam_breaks(n_scenes, seed=seed, count_range=(300, 4000))
    for p, _, _, _ in sc:
        p.boundary_pressure_mode = mode
    return sc


def _plain(scenes, nsteps):
    out = []
    for p, pos, typ, nf in scenes:
        sim = upf.Simulation(p, len(typ))
        sim.upload(pos, typ)
        sim.step(nsteps, upf.UPF_PCISPH_STATIC)
        st = sim.state()
        K, r = sim.stats()
        out.append((st, K, r))
        sim.close()
    return out


def _split(scenes, arr):
    offs = np.cumsum([0] + [len(s[2]) for s in scenes])
    return [arr[offs[k]:offs[k + 1]] for k in range(len(scenes))]


@pytest.mark.parametrize("use_graph", [1, 0, 2])
@pytest.mark.parametrize("mode", [upf.UPF_BOUNDARY_CPU_REF, upf.UPF_BOUNDARY_AKINCI])
def test_batch_equals_plain_per_scene(gpu, use_graph, mode):
    nsteps = 6
    scenes = _scenes(mode=mode)
    print("batch vs plain: %d scenes, counts %s, graph=%s mode=%d" %
          (len(scenes), [len(s[2]) for s in scenes], use_graph, mode), flush=True)
    ref = _plain(scenes, nsteps)
    b = upf.Batch.from_scenes(scenes)
    b.step(nsteps, use_graph=use_graph)
    st = b.state()
    K, r = b.stats()
    b.close()
    assert K.shape == (nsteps, len(scenes))
    for k, (pos, vel, rho) in enumerate(zip(_split(scenes, st["pos"]), _split(scenes, st["vel"]),
                                            _split(scenes, st["rho"]))):
        g, Kp, rp = ref[k]
        f = scenes[k][2] == upf.UPF_LIQUID
        assert np.array_equal(pos[:, :3], g["pos"][:, :3]), "scene %d positions" % k
        assert np.array_equal(vel[:, :3], g["vel"][:, :3]), "scene %d velocities" % k
        assert np.array_equal(rho[f], g["rho"][f]), "scene %d densities" % k
        assert list(K[:, k]) == list(Kp), "scene %d iteration counts" % k
        assert np.array_equal(r[:, k], rp), "scene %d max densities" % k


def test_batch_graph_repeated_calls_and_oracle(gpu):
    """Graph replays over several calls (both slot buffers), one scene checked
    against the oracle directly."""
    scenes = _scenes(n_scenes=4, seed=5)
    b = upf.Batch.from_scenes(scenes)
    b.step(1, use_graph=True)
    b.step(2, use_graph=True)
    b.step(3, use_graph=True)
    st = b.state()
    K, _ = b.stats()
    b.close()
    p, pos, typ, nf = scenes[2]
    o = ol.OracleSim(p, pos, None, typ)
    o.step(6, upf.UPF_PCISPH_STATIC)
    r = o.state()
    mine = _split(scenes, st["pos"])[2]
    assert np.array_equal(mine[:, :3], r["pos"][:, :3])
    Ko, _ = o.stats()
    assert list(K[:, 2]) == list(Ko)


def test_batch_rejects_mixed_physics(gpu):
    scenes = _scenes(n_scenes=2)
    p0, p1 = scenes[0][0].copy(), scenes[1][0].copy()
    p1.visc_const = p1.visc_const * 2
    with pytest.raises(upf.UPFError):
        upf.Batch([p0, p1], [len(scenes[0][2]), len(scenes[1][2])])


@pytest.mark.parametrize("mode", [upf.UPF_BOUNDARY_CPU_REF, upf.UPF_BOUNDARY_AKINCI])
def test_single_scene_graph_equals_plain(gpu, mode):
    """A plain scene replayed as a hipGraph (a batch of one) steps exactly like upf_step."""
    p, pos, typ, nf = upf.standard_dam_break(14, 10, 12, seed=3)
    p.boundary_pressure_mode = mode
    print("single-scene graph: %d particles mode=%d" % (len(typ), mode), flush=True)
    sim = upf.Simulation(p, len(typ))
    sim.upload(pos, typ)
    sim.step(7, upf.UPF_PCISPH_STATIC)
    g = sim.state()
    Kp, rp = sim.stats()
    sim.close()
    b = upf.Batch([p], [len(typ)])
    b.upload(pos, typ)
    b.step(3, use_graph=True)
    b.step(4, use_graph=True)
    st = b.state()
    K, r = b.stats()
    b.close()
    assert np.array_equal(st["pos"][:, :3], g["pos"][:, :3])
    assert np.array_equal(st["vel"][:, :3], g["vel"][:, :3])
    assert list(K[:, 0]) == list(Kp)
    assert np.array_equal(r[:, 0], rp)


@pytest.mark.parametrize("use_graph", [True, False])
def test_batch_with_union_lists_equals_plain(gpu, use_graph):
    """The batch with the correction loop on per-chunk unions (loop_list 2:
    chunks of 256 slots that cross scene boundaries) equals the plain
    per-scene runs, graph-replayed or not."""
    from unifiedparticleframeworkcuda_amd import autotune
    nsteps = 5
    scenes = _scenes(seed=13)
    ref = _plain(scenes, nsteps)
    b = upf.Batch.from_scenes(scenes)
    b.set_tuning(dict(autotune.DEFAULT, loop_list=2))
    b.step(nsteps, use_graph=use_graph)
    st = b.state()
    b.close()
    for k, (pos, vel) in enumerate(zip(_split(scenes, st["pos"]), _split(scenes, st["vel"]))):
        g = ref[k][0]
        assert np.array_equal(pos[:, :3], g["pos"][:, :3]), "scene %d positions" % k
        assert np.array_equal(vel[:, :3], g["vel"][:, :3]), "scene %d velocities" % k


def test_batch_graph_follows_set_params(gpu):
    """upf_set_params on the batch's simulation handle after the step graph
    was captured (a shorter time step, fewer loop iterations): the graph is
    recaptured, so graph replays give exactly what the host-loop batch gives."""
    scenes = _scenes(n_scenes=3, seed=9)
    out = []
    for use_graph in (1, 0, 2):
        b = upf.Batch.from_scenes(scenes)
        b.step(2, use_graph=use_graph)  # the graph is captured here
        q = scenes[0][0].copy()
        q.dt = 0.0008
        q.max_loops = 7
        upf.check("upf_set_params", upf.lib().upf_set_params(b.sim_handle(), C.byref(q)))
        b.step(3, use_graph=use_graph)
        st = b.state()
        K, r = b.stats()
        out.append((st, K, r))
        b.close()
    (a, Ka, ra) = out[1]
    for g, Kg, rg in (out[0], out[2]):
        assert np.array_equal(a["pos"], g["pos"]) and np.array_equal(a["vel"], g["vel"])
        assert np.array_equal(Ka, Kg) and np.array_equal(ra, rg)
    assert Ka[2:].max() <= 7


@pytest.mark.parametrize("use_graph", [1, 0, 2])
def test_batch_with_a_crowded_cell_equals_plain(gpu, use_graph):
    """A pile of wall particles in one scene's cell: the sort by blocks of the first call, graphs captured with it
    and graphs captured again with the radix sort give the plain per-scene runs."""
    import scenes as sc
    some = _scenes(n_scenes=3, seed=4)
    some[1] = (some[1][0],) + sc.with_pile(*some[1][:3], 7000)
    print("crowded batch: counts %s, graph %s" % ([len(s[2]) for s in some], use_graph), flush=True)
    b = upf.Batch.from_scenes(some)
    for steps in (2, 2, 3):
        b.step(steps, use_graph=use_graph)
    st = b.state()
    b.close()
    off = 0
    for p, pos, typ in (s[:3] for s in some):
        sim = upf.Simulation(p, len(typ))
        sim.upload(pos, typ)
        sim.step(7, upf.UPF_PCISPH_STATIC)
        r = sim.state()
        sim.close()
        for k in ("pos", "vel", "rho"):
            assert np.array_equal(st[k][off:off + len(typ)], r[k]), k
        off += len(typ)
