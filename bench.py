"""Benchmark: PCISPH particle-updates/s of the 1M-particle dam break on one MI355X.

Workload (the metric's configuration): 128 x 64 x 128 = 1,048,576 fluid
particles (spacing 0.01 m, jitter +-0.001 spacing, seed 0) in the corner of a
2.56 x 0.64 x 1.28 m box with one layer of wall particles at the spacing
(~84k), PCISPH with min 3 / max 50 iterations and a 1 % density-error
threshold, Morton sort every step, dt = 1 ms, FP32.  One particle-update =
one fluid particle advanced one full step including all K iterations.  A
second leg (`half_spacing_walls`) runs the same fluid in the wall layout the
configuration names -- walls sampled at half the spacing (~335k boundary
particles) -- with Akinci boundary volumes.

Prints ONE JSON line.  `roofline` is for the kernel class with the largest
device time (HIP events recorded by the library on its own stream around every
launch during the timed steps); `cpu_baseline` times the CPU oracle (OpenMP
port of the reference CPU path) on a bounded sample of the same workload.
"""
import argparse
import ctypes as C
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK = 8.0e12  # MI355X HBM3E bytes/s


def step_bytes(n, nf, ncells, k):
    """Algorithmic bytes of one step at K iterations (compulsory traffic:
    each SoA field a pass touches once per pass; neighbour re-reads on chip).
    key 20N, sort 12N, reorder 76N, cell table 4N + 8C, external forces
    40N + 36N_f, per iteration predict 80N_f + density 16N + 12N_f + force
    20N + 16N_f, integrate 96N_f."""
    return 152 * n + 132 * nf + 8 * ncells + k * (36 * n + 108 * nf)


# Algorithmic bytes per launch of each kernel class, from the same model.
def class_bytes(name, n, nf, ncells):
    table = {
        "radix_sort": 12 * n + 20 * n,          # (by cells or by key) key read + (key, perm) write, keys from integration
        "gather": 76 * n,
        "cell_table": 4 * n + 8 * ncells,
        "neighbour_lists": 20 * n + 4 * n,      # positions + keys read, counts written
        "external_force_predict": 40 * n + 36 * nf + 80 * nf,  # + the fused first prediction
        "neighbour_lists_external_force": 24 * n + 40 * n + 36 * nf + 80 * nf,  # both in one kernel
        "predicted_density": 16 * n + 12 * nf,
        "pressure_force_predict": 20 * n + 16 * nf + 80 * nf,  # + the fused next prediction
        "integrate": 96 * nf,
    }
    return table.get(name)


# kernel symbol prefix of each profile class of the default path (for the
# committed PMC summary; the separate list build and external-force kernels
# of nbr_fuse 0 have no row there)
CLASS_KERNEL = {"pressure_force_predict": "upf::k_force<", "predicted_density": "upf::k_density<",
                "neighbour_lists_external_force": "upf::k_nbr_build_ext<",
                "integrate": "upf::k_integrate", "gather": "upf::k_rank_gather"}
PROFILE = os.path.join(ROOT, "profiles", "pcisph_dam_break_1m_kernels.md")


def measured_traffic(cls):
    """HBM bytes per launch of the class's kernel from the committed rocprofv3
    counter summary (FETCH_SIZE + WRITE_SIZE, scaled by a copy of known size),
    or None when the summary has no row for it."""
    pre = CLASS_KERNEL.get(cls)
    if pre is None or not os.path.exists(PROFILE):
        return None
    in_table = False
    for line in open(PROFILE):
        if line.startswith("| kernel |"):
            # the traffic table: | kernel | dispatches | fetch MB | write MB | total MB |
            in_table = "total MB" in line
            continue
        if in_table and line.startswith("| " + pre):
            cells = [c.strip() for c in line.strip().strip("|").split("|")]
            if len(cells) == 5:
                return float(cells[4]) * 1e6
    return None


# The dam-break workloads: wall sampling (relative to the spacing) and the
# boundary-pressure mode.
WORKLOADS = {
    # one wall layer at the full spacing (~84k) with the CPU path's boundary
    # pressure (whose Akinci term is zero): the walls act through the density
    "pcisph_dam_break_1m": dict(wall_rel=1.0, mode="cpu_ref"),
    # the configuration's wall layout: walls sampled at half spacing (~335k)
    # with Akinci boundary volumes (the reference GPU path's boundary pressure;
    # with the CPU path's fluid mass such walls would weigh four layers)
    "pcisph_dam_break_1m_half_spacing_walls": dict(wall_rel=0.5, mode="akinci"),
}


def build_scene(name, lattice):
    """(params, pos4, type, n_fluid) of a dam-break workload."""
    import unifiedparticleframeworkcuda_amd as upf
    nx, ny, nz = lattice
    w = WORKLOADS[name]
    p = upf.make_params(0.01, 0.001)
    pos, typ, nf = upf.dam_break(p, nx, ny, nz, (0.02 * nx, 0.01 * ny, 0.01 * nz), wall_rel=w["wall_rel"])
    upf.density_error_factor(p)
    p.boundary_pressure_mode = upf.UPF_BOUNDARY_AKINCI if w["mode"] == "akinci" else upf.UPF_BOUNDARY_CPU_REF
    return p, pos, typ, nf


def loop_summary(K, rmax, max_loops=50):
    """Iteration counts and density errors of a run's steps: the loop stops
    once the largest predicted density is within 1 % of rho0 (after at least
    3 iterations) or after max_loops; steps that reach max_loops end above."""
    K = np.asarray(K)
    err = np.maximum(0.0, 0.1 * np.asarray(rmax, np.float64) - 100.0)
    conv = K < max_loops
    return {"iterations": {"mean": float(np.mean(K)), "max": int(np.max(K)),
                           "hist": {str(int(k)): int(c) for k, c in zip(*np.unique(K, return_counts=True))}},
            "steps_at_max_loops": int(np.sum(~conv)),
            "max_density_error_pct": float(err.max()),
            "max_density_error_pct_converged_steps": float(err[conv].max()) if conv.any() else None}


def run_gpu(args, workload=None, steps=None, profile=True):
    import unifiedparticleframeworkcuda_amd as upf
    workload = workload or args.workload
    steps = steps or args.steps
    nx, ny, nz = args.lattice
    p, pos, typ, nf = build_scene(workload, args.lattice)
    n = len(typ)
    sim = upf.Simulation(p, n)
    tuning = None
    if args.tuning:
        tuning = dict(sim.tuning().as_dict(), **json.loads(args.tuning))
        sim.set_tuning(tuning)
    elif not args.no_tune:
        from unifiedparticleframeworkcuda_amd import autotune
        trials = []
        tuning, tune_ms = autotune.tune_simulation(sim, pos, typ, "%s_%dx%dx%d" % (workload, nx, ny, nz),
                                                   use_cache=not args.retune, log=trials)
        if args.show_trials:
            for t, sec in trials:
                print("tuning trial %s: %.3f ms" % (t, sec * 1e3), file=sys.stderr)
    if args.no_speculate:
        sim.set_tuning(dict(sim.tuning().as_dict(), speculate=1, spec_first=0))
    L = upf.lib()
    # The library links the system HIP runtime; torch bundles its own, and the
    # two do not share one process, so the device is synchronised through the
    # library's runtime (upf_step also returns only after its stream drained).
    hip = C.CDLL("libamdhip64.so")
    # timed run: no event recording
    sim.upload(pos, typ)
    sim.step(args.warmup, upf.UPF_PCISPH_STATIC)
    hip.hipDeviceSynchronize()
    t0 = time.perf_counter()
    sim.step(steps, upf.UPF_PCISPH_STATIC)
    hip.hipDeviceSynchronize()
    dt = time.perf_counter() - t0
    K, rmax = sim.stats()
    Kt = K[-steps:]
    rt = rmax[-steps:]
    keys, ids, cells = sim.sorted_state()
    ncells = len(cells)
    if not profile:
        sim.close()
        return dict(p=p, n=n, nf=nf, ncells=ncells, seconds=dt, K=Kt, rmax=rt, tuning=tuning)
    # the same steps again (same inputs, same iteration counts) with HIP events
    # recorded around every launch: per-kernel-class device time.  Here the
    # host enqueues no iteration ahead of the loop decision, so that every
    # launch of the iteration passes does work (launch shapes unchanged).
    # The kernels of a step run back to back, so their device times should
    # add up to the timed run's step time; a replay whose event times fall
    # short of it by more than 1.5 % (seen now and then) is run again, up to
    # three times, and the replay with the largest sum is kept (the most
    # conservative per-kernel times).
    timed_tuning = sim.tuning().as_dict()
    sim.set_tuning(dict(timed_tuning, speculate=1, spec_first=0))
    best = None
    for attempt in range(1, 4):
        sim.upload(pos, typ)
        sim.step(args.warmup, upf.UPF_PCISPH_STATIC)
        L.upf_profile_enable(sim.h, 1)
        L.upf_profile_reset(sim.h)
        hip.hipDeviceSynchronize()
        t0 = time.perf_counter()
        sim.step(steps, upf.UPF_PCISPH_STATIC)
        hip.hipDeviceSynchronize()
        replay_s = time.perf_counter() - t0
        Kp, _ = sim.stats()
        prof = upf.profile(sim.h)
        L.upf_profile_enable(sim.h, 0)
        assert np.array_equal(Kp[-steps:], Kt), "the profiled replay took other iteration counts"
        total = sum(v[0] for v in prof.values()) * 1e-3
        if best is None or total > best[0]:
            best = (total, prof, replay_s, attempt)
        if total >= 0.985 * dt:
            break
    _, prof, replay_s, _ = best
    sim.set_tuning(timed_tuning)
    sim.close()
    out = dict(p=p, n=n, nf=nf, ncells=ncells, seconds=dt, K=Kt, rmax=rt, prof=prof, tuning=tuning,
               replay_seconds=replay_s, replay_attempts=attempt)
    if not args.no_graph:
        # the same scene as a batch of one: every step one hipGraph replay
        b = upf.Batch([p], [n], max_record_steps=args.warmup + steps + 8)
        if tuning:
            b.set_tuning(tuning)
        b.upload(pos, typ)
        b.step(args.warmup, use_graph=True)
        hip.hipDeviceSynchronize()
        t0 = time.perf_counter()
        b.step(steps, use_graph=True)
        hip.hipDeviceSynchronize()
        out["graph_seconds"] = time.perf_counter() - t0
        Kg, _ = b.stats()
        out["graph_K"] = Kg[-steps:, 0]
        b.close()
    return out


def copy_calibration(nbytes=1 << 28):
    """A device-to-device copy of known size (the runtime's copy kernel), so
    that hardware byte counters can be scaled: FETCH_SIZE / WRITE_SIZE of this
    dispatch should read nbytes each."""
    hip = C.CDLL("libamdhip64.so")
    a, b = C.c_void_p(), C.c_void_p()
    assert hip.hipMalloc(C.byref(a), C.c_size_t(nbytes)) == 0
    assert hip.hipMalloc(C.byref(b), C.c_size_t(nbytes)) == 0
    hip.hipMemset(a, 1, C.c_size_t(nbytes))
    for _ in range(3):
        hip.hipMemcpy(b, a, C.c_size_t(nbytes), 3)  # hipMemcpyDeviceToDevice
    hip.hipDeviceSynchronize()
    hip.hipFree(a)
    hip.hipFree(b)


def run_batch(args):
    """256 uneven dam breaks (fluid counts log-uniform in [2048, 65536], block
    aspect ratios in [0.5, 2], own box and walls each): the batched form
    (one launch per stage for all scenes) with every step one whole-loop
    hipGraph replay, with split graphs (head, chunks of iterations, tail;
    the loop decision read back between them) and with the host loop, each
    from the same initial state over the same steps (same iteration counts,
    asserted), against the plain path (one simulation per scene, upf_step
    per scene), same scenes, same steps."""
    import unifiedparticleframeworkcuda_amd as upf
    hip = C.CDLL("libamdhip64.so")
    scenes = upf.batch_dam_breaks(args.batch_scenes, seed=0)
    nf = sum(sc[3] for sc in scenes)
    n = sum(len(sc[2]) for sc in scenes)
    K = args.batch_steps
    out = dict(scenes=len(scenes), fluid=nf, particles=n, steps=K)
    allpos = np.concatenate([sc[1] for sc in scenes])
    alltyp = np.concatenate([sc[2] for sc in scenes])
    b = upf.Batch.from_scenes(scenes, max_record_steps=K + 64)
    if not args.no_tune:
        from unifiedparticleframeworkcuda_amd import autotune
        bt, _ = autotune.tune_batch(b, allpos, alltyp, "batch_%d_scenes_seed0" % len(scenes),
                                    use_cache=not args.retune)
        out["tuning"] = bt
    t = {}
    Ks = rs = None
    for name, mode in (("graph", 1), ("graph_split", 2), ("host_loop", 0)):
        b.upload(allpos, alltyp)
        b.step(2, use_graph=mode)  # eager first step (boundary volumes), graph capture + one replay
        hip.hipDeviceSynchronize()
        t0 = time.perf_counter()
        b.step(K, use_graph=mode)
        hip.hipDeviceSynchronize()
        t[name] = time.perf_counter() - t0
        Km, rm = b.stats()
        if Ks is None:
            Ks, rs = Km, rm
        elif not (np.array_equal(Km, Ks) and np.array_equal(rm, rs)):
            raise RuntimeError("batched modes disagree on the loop statistics")
    b.close()
    tg, ts, th = t["graph"], t["graph_split"], t["host_loop"]
    sims = []
    for p, pos, typ, _ in scenes:
        s = upf.Simulation(p, len(typ))
        s.upload(pos, typ)
        s.step(2, upf.UPF_PCISPH_STATIC)
        sims.append(s)
    hip.hipDeviceSynchronize()
    t0 = time.perf_counter()
    for s in sims:
        s.step(K, upf.UPF_PCISPH_STATIC)
    hip.hipDeviceSynchronize()
    tp = time.perf_counter() - t0
    for s in sims:
        s.close()
    # the byte model summed over scenes, each at its own iteration count
    KK = np.asarray(Ks[2:2 + K])
    model = sum(step_bytes(len(sc[2]), sc[3], int(sc[0].grid_dim) ** 3, int(KK[:, j].sum()) / K) * K
                for j, sc in enumerate(scenes))
    best = min(tg, ts, th)
    out["byte_model"] = {"bytes_per_step": model / K, "achieved": model / best / 1e9, "unit": "GB/s",
                         "frac": model / best / HBM_PEAK, "mode": min(t, key=t.get)}
    out.update(graph_updates_per_s=nf * K / tg, graph_split_updates_per_s=nf * K / ts,
               host_loop_updates_per_s=nf * K / th, plain_updates_per_s=nf * K / tp,
               graph_ms_per_step=tg / K * 1e3, graph_split_ms_per_step=ts / K * 1e3,
               host_loop_ms_per_step=th / K * 1e3, plain_ms_per_step=tp / K * 1e3,
               speedup_graph_vs_plain=tp / tg, speedup_graph_split_vs_plain=tp / ts,
               iterations_mean=float(np.mean(Ks[2:2 + K])),
               iterations_max=int(np.max(Ks[2:2 + K])),
               max_density_error_pct=float(max(0.0, 0.1 * float(np.max(rs[2:2 + K])) - 100.0)))
    return out


def run_adjoint(args):
    """The gradient workload: 65,536-particle dam break (64x32x32 lattice),
    64 steps of 5 iterations, checkpoint every 8 steps; gradient of the mean
    squared distance to a target cloud with respect to the initial
    velocities.  Device time of the forward and of the backward pass."""
    from unifiedparticleframeworkcuda_amd import adjoint as adj
    p, pos, typ, vel, target, f = adj.differentiable_dam_break()
    r = adj.Rollout(p, pos, typ, 64, 5, checkpoint_every=8)
    best = None
    for _ in range(3):
        x, _ = r.forward(vel)
        g = np.zeros_like(x)
        g[f] = 2.0 * (x[f] - target[f]) / f.sum()
        r.backward(g)
        fwd, bwd, mem = r.timing()
        if best is None or fwd + bwd < best[0] + best[1]:
            best = (fwd, bwd, mem)
    r.close()
    fwd, bwd, mem = best
    return dict(particles=len(typ), fluid=int(f.sum()), steps=64, iterations=5, checkpoint_every=8,
                forward_ms=fwd, backward_ms=bwd, backward_over_forward=bwd / fwd, device_mb=mem / 1e6,
                forward_updates_per_s=int(f.sum()) * 64 / (fwd / 1e3))


def _timed_steps(sim, steps, method):
    hip = C.CDLL("libamdhip64.so")
    hip.hipDeviceSynchronize()
    t0 = time.perf_counter()
    sim.step(steps, method)
    hip.hipDeviceSynchronize()
    return time.perf_counter() - t0


def run_wcsph(args):
    """The WCSPH variant on the same 1M inputs: Tait EOS, stiffness 1000,
    gamma 7, at the CFL step 0.4 h / c = 0.253 ms; the 1 ms step of the
    PCISPH runs is also tried (it violates the CFL condition).  Also the
    original SPH (linear EOS, k = 1000) at 0.253 ms ("sph_...")."""
    import unifiedparticleframeworkcuda_amd as upf
    nx, ny, nz = args.lattice
    out = {}
    for method, dt, steps in ((upf.UPF_WCSPH_STATIC, 0.000253, 20), (upf.UPF_WCSPH_STATIC, 0.001, 20),
                              (upf.UPF_SPH_STATIC, 0.000253, 20)):
        p, pos, typ, nf = upf.standard_dam_break(nx, ny, nz, dt=dt)
        p.gas_const_wcsph = 1000.0
        sim = upf.Simulation(p, len(typ))
        sim.upload(pos, typ)
        key = ("sph_" if method == upf.UPF_SPH_STATIC else "") + "dt_%gms" % (dt * 1e3)
        try:
            sim.step(3, method)
            sec = _timed_steps(sim, steps, method)
            st = sim.state()
            f = typ == upf.UPF_LIQUID
            out[key] = {"updates_per_s": nf * steps / sec, "ms_per_step": sec / steps * 1e3, "stable": True,
                        "max_speed": float(np.max(np.linalg.norm(st["vel"][f, :3], axis=1))),
                        "max_density_error_pct": float(max(0.0, (np.max(st["rho"][f]) - 1000.0) / 10.0))}
        except upf.UPFError as e:
            out[key] = {"stable": False, "error": str(e)}
        sim.close()
    return out


def run_wall_weight(args):
    """PCISPH on the 1M dam break's fluid without its wall particles, the
    container's walls entering the predicted density through the wall weight
    function (add_wall_weight), against the same steps without it: ms per
    step and per correction iteration (the term costs one distance and six
    table reads per liquid particle and iteration)."""
    import unifiedparticleframeworkcuda_amd as upf
    nx, ny, nz = args.lattice
    out = {}
    for on in (1, 0):
        p, pos, typ, nf = upf.standard_dam_break(nx, ny, nz)
        f = typ == upf.UPF_LIQUID
        pos, typ = pos[f], typ[f]
        p.add_wall_weight = on
        sim = upf.Simulation(p, len(typ))
        sim.upload(pos, typ)
        sim.step(3, upf.UPF_PCISPH_STATIC)
        steps = 20
        sec = _timed_steps(sim, steps, upf.UPF_PCISPH_STATIC)
        K, rmax = sim.stats()
        sim.close()
        k = float(np.mean(K[-steps:]))
        out["on" if on else "off"] = {"ms_per_step": sec / steps * 1e3, "iterations_mean": k,
                                      "ms_per_iteration": sec / steps * 1e3 / k,
                                      "updates_per_s": nf * steps / sec,
                                      "max_density_error_pct": float(max(0.0, 0.1 * float(np.max(rmax[-steps:])) - 100.0))}
    return out


def run_rigid(args):
    """Rigid-fluid coupling: 524,288 fluid particles (64 x 128 x 64 block),
    64 seeded boxes and spheres sampled at half spacing, Akinci boundary
    volumes, surface tension 0.05, adhesion 0.01."""
    import unifiedparticleframeworkcuda_amd as upf
    p, pos, typ, bid, rel, bodies, counts = upf.standard_rigid_scene(64, 128, 64, n_bodies=64)
    # the scene set-up's solidification of the same rigid particles (host)
    r = typ == upf.UPF_RIGID
    t0 = time.perf_counter()
    built = upf.bodies_from_particles(p, pos[r], rel[r, 3])
    build_ms = (time.perf_counter() - t0) * 1e3
    sim = upf.Simulation(p, len(typ))
    sim.upload(pos, typ)
    sim.upload_bodies(bodies, bid, rel)
    sim.step(3, upf.UPF_PCISPH_RIGID)
    steps = 10
    sec = _timed_steps(sim, steps, upf.UPF_PCISPH_RIGID)
    K, rmax = sim.stats()
    sim.close()
    nf, nr, nw = counts
    return {"fluid": nf, "rigid_particles": nr, "wall": nw, "bodies": 64, "steps": steps,
            "updates_per_s": nf * steps / sec, "ms_per_step": sec / steps * 1e3,
            "iterations_mean": float(np.mean(K[-steps:])),
            "bodies_from_particles": {"particles": int(r.sum()), "bodies": len(built[2]), "ms": build_ms}}


def run_model_fill(args):
    """OBJ model -> particles (ObjectLoader::LoadParticles): a procedural
    non-convex blob of 6,400 triangles written as OBJ, read with the
    reference's reader, filled at the bunny placement's scale 2.5 with spacing
    0.005 (1.4M lattice points) on the GPU; the oracle (single thread) fills the
    same mesh at spacing 0.02 as its bounded sample.  Rate = lattice-point x
    face tests per second."""
    import tempfile
    import unifiedparticleframeworkcuda_amd as upf
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import meshes
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "blob.obj")
        with open(path, "w") as f:
            f.write(meshes.sphere(0.08, 80, 41, center=(-0.05, 0.1, 0.04), bump=0.25, seed=3))
        faces = upf.load_obj(path)
    nf = len(faces)
    mn = np.minimum(faces.reshape(-1, 3).min(0), 0.0)
    mx = np.maximum(faces.reshape(-1, 3).max(0), 0.0)

    def lattice(sp):
        steps = (mx - mn).astype(np.float32) * np.float32(2.5) / np.float32(sp)
        return int(np.prod(np.floor(steps) + 1))

    sp = 0.005
    upf.mesh_fill(faces, 2.5, sp)  # warm-up (module load, first allocation)
    reps = 3
    t0 = time.perf_counter()
    for _ in range(reps):
        pos = upf.mesh_fill(faces, 2.5, sp)
    gpu_s = (time.perf_counter() - t0) / reps
    out = {"faces": nf, "lattice_points": lattice(sp), "particles": int(len(pos)), "spacing": sp, "scale": 2.5,
           "gpu_ms": gpu_s * 1e3, "gpu_tests_per_s": lattice(sp) * nf / gpu_s}
    if not args.no_cpu:
        import oracle_lib as ol
        csp = 0.02
        t0 = time.perf_counter()
        cpos = ol.mesh_fill(faces, 2.5, csp)
        cpu_s = time.perf_counter() - t0
        out["cpu_oracle"] = {"spacing": csp, "lattice_points": lattice(csp), "particles": int(len(cpos)),
                             "seconds": cpu_s, "tests_per_s": lattice(csp) * nf / cpu_s, "threads": 1}
        out["speedup_tests_per_s"] = out["gpu_tests_per_s"] / out["cpu_oracle"]["tests_per_s"]
    return out


def run_state_io(args):
    """Particle state files of the 1M dam break after 5 steps (the reference's
    UnifiedIO, src/cpu/UnifiedIO.cpp): the restart file written from the
    device (upf_save_text: download + formatting on up to 16 host threads),
    read back (upf_read_restart) and uploaded (upf_upload_restart), and the
    liquid dump SaveLiquidParticleInfoFull writes.  CPU leg: the oracle's
    iostream writer and reader (one thread, the reference's formatting) on
    the same particles."""
    import filecmp
    import tempfile
    import unifiedparticleframeworkcuda_amd as upf
    nx, ny, nz = args.lattice
    p, pos, typ, nf = upf.standard_dam_break(nx, ny, nz)
    sim = upf.Simulation(p, len(typ))
    sim.upload(pos, typ)
    sim.step(5, upf.UPF_PCISPH_STATIC)
    n = len(typ)
    with tempfile.TemporaryDirectory() as d:
        rpath, lpath = os.path.join(d, "restart.txt"), os.path.join(d, "liquid.txt")
        t0 = time.perf_counter()
        sim.save_text(rpath, upf.UPF_TEXT_RESTART)
        t_save = time.perf_counter() - t0
        size = os.path.getsize(rpath)
        t0 = time.perf_counter()
        st = upf.read_restart(rpath)
        t_read = time.perf_counter() - t0
        t0 = time.perf_counter()
        sim.upload_restart(st)
        t_up = time.perf_counter() - t0
        t0 = time.perf_counter()
        sim.save_text(lpath, upf.UPF_TEXT_LIQUID)
        t_liq = time.perf_counter() - t0
        out = {"particles": n, "restart_bytes": size, "save_restart_ms": t_save * 1e3, "read_restart_ms": t_read * 1e3,
               "upload_restart_ms": t_up * 1e3, "save_liquid_ms": t_liq * 1e3,
               "liquid_bytes": os.path.getsize(lpath), "save_restart_MBps": size / t_save / 1e6,
               "read_restart_MBps": size / t_read / 1e6}
        if not args.no_cpu:
            sys.path.insert(0, os.path.join(ROOT, "tests"))
            import oracle_lib as ol
            opath = os.path.join(d, "oracle.txt")
            t0 = time.perf_counter()
            ol.write_text(opath, upf.UPF_TEXT_RESTART, st["pos"], st["type"], st["vel"], st["corr_pressure"],
                          st["predicted_density"])
            t_ow = time.perf_counter() - t0
            t0 = time.perf_counter()
            ol.read_restart(opath, cap=n)
            t_or = time.perf_counter() - t0
            out["cpu_oracle"] = {"write_ms": t_ow * 1e3, "read_ms": t_or * 1e3, "threads": 1,
                                 "same_bytes": filecmp.cmp(opath, rpath, shallow=False)}
    sim.close()
    return out


def cpu_baseline(args, budget_s):
    """The oracle (OpenMP C++ port of the reference CPU path) on the same
    workload: steps until the time budget is used (at least one)."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib as ol
    import unifiedparticleframeworkcuda_amd as upf
    p, pos, typ, nf = build_scene(args.workload, args.lattice)
    o = ol.OracleSim(p, pos, None, typ, omp=True)
    steps = 0
    t0 = time.perf_counter()
    while True:
        o.step(1, upf.UPF_PCISPH_STATIC)
        steps += 1
        el = time.perf_counter() - t0
        if el >= budget_s or steps >= args.cpu_max_steps:
            break
    threads = ol.oracle(True).orc_num_threads()
    out = dict(value=nf * steps / el, unit="particle-updates/s", cores=int(threads), kind="port",
               sample="first %d step(s) of the same 1M dam break (%s) from its initial state, %.1f s" % (steps, args.workload, el))
    try:
        with open("/proc/cpuinfo") as f:
            out["cpu_model"] = next(l.split(":", 1)[1].strip() for l in f if l.startswith("model name"))
    except (OSError, StopIteration):
        pass
    if args.cpu_single_steps > 0:
        # the same first step(s) on one thread (the oracle's serial build)
        o1 = ol.OracleSim(p, pos, None, typ, omp=False)
        t0 = time.perf_counter()
        o1.step(args.cpu_single_steps, upf.UPF_PCISPH_STATIC)
        el1 = time.perf_counter() - t0
        out["single_thread"] = {"value": nf * args.cpu_single_steps / el1, "cores": 1,
                                "sample": "first %d step(s), %.1f s" % (args.cpu_single_steps, el1)}
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--lattice", type=int, nargs=3, default=[128, 64, 128])
    ap.add_argument("--workload", default="pcisph_dam_break_1m", choices=sorted(WORKLOADS))
    ap.add_argument("--no-second-layout", action="store_true",
                    help="skip the leg with the other wall layout")
    ap.add_argument("--cpu-budget", type=float, default=15.0)
    ap.add_argument("--cpu-max-steps", type=int, default=20)
    ap.add_argument("--cpu-single-steps", type=int, default=1, help="steps of the single-thread CPU sample (0: none)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--batch-scenes", type=int, default=256)
    ap.add_argument("--batch-steps", type=int, default=10)
    ap.add_argument("--no-batch", action="store_true")
    ap.add_argument("--no-graph", action="store_true")
    ap.add_argument("--no-adjoint", action="store_true")
    ap.add_argument("--no-wcsph", action="store_true")
    ap.add_argument("--no-rigid", action="store_true")
    ap.add_argument("--no-model-fill", action="store_true")
    ap.add_argument("--no-state-io", action="store_true")
    ap.add_argument("--no-wall-weight", action="store_true")
    ap.add_argument("--no-tune", action="store_true", help="default launch shapes, no autotuning")
    ap.add_argument("--tuning", default=None,
                    help="launch shapes as JSON (fields of upf_tuning; the rest default), instead of autotuning")
    ap.add_argument("--retune", action="store_true", help="ignore the tuning cache")
    ap.add_argument("--show-trials", action="store_true", help="print every tuning trial to stderr")
    ap.add_argument("--no-speculate", action="store_true",
                    help="host loop enqueues no iteration ahead of the loop decision (every iteration-pass "
                         "launch does work; for kernel profiles)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="also run a 256 MiB device copy (scale for hardware byte counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py runs on one GPU only: the workload is one scene on one MI355X "
              "(how the step would shard over several GPUs is a design note only)", file=sys.stderr)
        sys.exit(2)
    if args.copy_calibration:
        copy_calibration()
    g = run_gpu(args)
    n, nf, ncells = g["n"], g["nf"], g["ncells"]
    sec = g["seconds"]
    value = nf * args.steps / sec
    total_bytes = sum(step_bytes(n, nf, ncells, int(k)) for k in g["K"])
    # dominant kernel class
    dom = max(g["prof"].items(), key=lambda kv: kv[1][0])
    name, (ms, cnt) = dom
    # iteration passes: the host loop enqueues iterations ahead of the loop
    # decision and those that are not needed return at once; their (short)
    # time stays in the class total, which is divided by the iterations that
    # ran -- the average of a working launch, stated conservatively
    working = int(np.sum(g["K"])) if name in ("predicted_density", "pressure_force_predict") else cnt
    avg_s = ms / working / 1e3
    b = class_bytes(name, n, nf, ncells)
    roof = dict(bound="hbm", kernel=name, launches=cnt, working_launches=working, avg_us=avg_s * 1e6,
                achieved=(b / avg_s / 1e9) if b else None, peak=HBM_PEAK / 1e9, unit="GB/s",
                frac=(b / avg_s / HBM_PEAK) if b else None, traffic=measured_traffic(name),
                algorithmic_bytes=b)
    out = {
        "metric": "PCISPH particle-updates/s @1M; batched vs plain at <=1% density error",
        "value": value,
        "unit": "particle-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": sec / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": args.workload, "fluid": nf, "boundary": n - nf,
                   "lattice": list(args.lattice), "spacing_m": 0.01, "dt_s": 0.001,
                   "wall_sampling_rel": WORKLOADS[args.workload]["wall_rel"],
                   "boundary_mode": WORKLOADS[args.workload]["mode"],
                   "min_max_iterations": [3, 50], "density_error_threshold_pct": 1.0, "path": "plain"},
        "step_roofline": {"achieved": total_bytes / sec / 1e9, "unit": "GB/s", "frac": total_bytes / sec / HBM_PEAK,
                          "bytes_per_update": total_bytes / (nf * args.steps)},
        "kernel_ms_per_step": {k: v[0] / args.steps for k, v in g["prof"].items()},
        "replay_ms_per_step": g["replay_seconds"] / args.steps * 1e3,
        "replay_attempts": g["replay_attempts"],
        "tuning": g["tuning"],
        "graph_replay": (None if "graph_seconds" not in g else
                         {"ms_per_step": g["graph_seconds"] / args.steps * 1e3,
                          "updates_per_s": nf * args.steps / g["graph_seconds"],
                          "same_iterations": bool(np.array_equal(g["graph_K"], g["K"]))}),
        "roofline": roof,
    }
    out.update(loop_summary(g["K"], g["rmax"]))
    if not args.no_second_layout:
        other = [w for w in sorted(WORKLOADS) if w != args.workload][0]
        g2 = run_gpu(args, workload=other, steps=min(args.steps, 20), profile=False)
        out["half_spacing_walls" if other.endswith("half_spacing_walls") else "walls_at_spacing"] = dict(
            workload=other, fluid=g2["nf"], boundary=g2["n"] - g2["nf"], steps=len(g2["K"]),
            ms_per_step=g2["seconds"] / len(g2["K"]) * 1e3, updates_per_s=g2["nf"] * len(g2["K"]) / g2["seconds"],
            **loop_summary(g2["K"], g2["rmax"]))
    if not args.no_batch:
        out["batched"] = run_batch(args)
    if not args.no_adjoint:
        out["adjoint"] = run_adjoint(args)
    if not args.no_wcsph:
        out["wcsph"] = run_wcsph(args)
    if not args.no_rigid:
        out["rigid"] = run_rigid(args)
    if not args.no_model_fill:
        out["model_fill"] = run_model_fill(args)
    if not args.no_state_io:
        out["state_io"] = run_state_io(args)
    if not args.no_wall_weight:
        out["wall_weight"] = run_wall_weight(args)
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(args, args.cpu_budget)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
