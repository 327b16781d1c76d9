"""Benchmark of the MDOODZ Newton-iteration grid path on one MI355X.

One step = one Newton-iteration unit over the whole grid:
StrainRateComponents -> NonNewtonianViscosityGrid -> EvaluateRHS ->
RheologicalOperators(0) -> Picard CSR values -> RheologicalOperators(1) ->
Jacobian CSR values -> RheologicalOperators(0) -> residual + norms,
everything resident in HBM (the CSR patterns are built once per boundary-
condition set, outside the timed region, as they are once per time step).

Workload: the three-layer lithosphere (wet quartzite / plagioclase /
olivine + Peierls, Maxwell elasticity, Drucker-Prager) at 2049 x 1025 cells,
seeded synthetic fields.  The metric is cell updates per second:
(Nx-1)(Nz-1) / time per unit.

Prints ONE JSON line.
"""
import argparse
import ctypes as C
import importlib.util
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))

# algorithmic HBM bytes per cell update of each stage (each listed array
# element read or written once; FP64 = 8 B, tags 1 B, equation numbers 4 B)
STAGES = ["strain_rates", "interp_guess", "rheology", "rhs", "dtensor_picard", "picard_values", "dtensor_jacobian",
          "jacobian_values", "dtensor_picard_2", "residual"]
# kernels of each stage (names as in the rocprofv3 kernel trace) for the
# launch shape (rheology threads, Picard rows, Jacobian rows per block).  An
# isotropic model takes the fused D pass: one launch writes the J = 1 tensor
# and the J = 0 components the Picard rows and the residual read, and the
# two J = 0 stages run nothing.
def stage_kernels(shape, learned=False, fused=True, net_in_rheology=True):
    """(learned mode: the network runs in the rheology kernels' prologue, the
    default, or in its own pass k_mlp_guess beside the interpolation)"""
    rh, pic, jac = shape

    def values(kind, rows, capa, capb):
        # 64-row blocks: the split pass (the listed general waves, then the
        # tag-free ones; its instance for grids above 2048 blocks)
        if rows == 64:
            return ["k_values_split<%d, %d, %d, %d>" % (kind, capa, capb, (6, 3)[kind])]
        if rows:
            return ["k_values_mom<%d, %d, %d, %d>" % (kind, rows, capa, capb)]
        return ["k_values_mom_direct<%d>" % kind, "k_values_cont"]

    separate = learned and not net_in_rheology
    prep = ["k_mlp_guess", "k_guess_vertices"] if separate else []
    # timed by stage, the right-hand sides and the D tensor are launches of
    # their own; a unit runs them as one (k_rhs_dtensor<2, true>)
    d0 = [] if fused else ["k_rhs_dtensor<0, false>"]
    d1 = ["k_rhs_dtensor<2, false>"] if fused else ["k_rhs_dtensor<1, false>"]
    net = "true" if learned and net_in_rheology else "false"
    return {"strain_rates": ["k_strain_tile<true>"],
            "interp_guess": prep,
            "rheology": ["k_rheo_fast<%d, true, %s, %d>" % (rh, net, part) for part in ((1, 2) if net == "true" else (0,))],
            "rhs": ["k_rhs_dtensor<-1, true>"],
            "dtensor_picard": d0,
            "picard_values": values(0, pic, 9, 2),
            "dtensor_jacobian": d1,
            "jacobian_values": values(1, jac, 21, 6),
            "dtensor_picard_2": d0,
            "residual": ["k_residual_tile", "k_norms_final_slots"]}


# The strain rates and the vertex interpolation of div_u, T, P, d and phi
# are one launch: reads u, v, T, P, d, phi (48 B) and four tags (4 B),
# writes div_u, exxd, ezzd, exz_n at the centroid and exz, exxd_s, ezzd_s,
# div_u_s, T_s, P_s, d_s, phi_s at the vertex (96 B) -- the 76 + 80 B of
# the two separate stages less the read of div_u; the network's separate
# guess pass (learned mode without the fused guess) has no byte count.
BYTES_PER_CELL = {"strain_rates": 148, "interp_guess": 0, "rheology": 730, "rhs": 160, "dtensor_picard": 114,
                  "picard_values": 340, "dtensor_jacobian": 330, "jacobian_values": 668, "dtensor_picard_2": 114,
                  "residual": 204}
# the fused D pass writes D11 (= D22) at the centroid and D33 at the vertex
# of the J = 0 tensor beside the J = 1 tensor (+16 B); the Picard values and
# the residual read that D11 once for D11 and D22 (-8 B each)
FUSED_BYTES_PER_CELL = dict(BYTES_PER_CELL, dtensor_picard=0, dtensor_jacobian=346, dtensor_picard_2=0,
                            picard_values=332, residual=196)
HBM_PEAK_GBS = 8000.0


def _pkg():
    spec = importlib.util.spec_from_file_location("mdoodz_amd", os.path.join(ROOT, "mdoodz6.0_amd", "__init__.py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules["mdoodz_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


def traffic_from_profile(kernels, ncx, ncz, mode):
    """HBM bytes per launch of a stage's kernels from the committed counter
    summary (FETCH_SIZE + WRITE_SIZE, scaled by the copy probe), or None."""
    path = os.path.join(ROOT, "profiles", "hbm_traffic_lithosphere_%dx%d_%s.md" % (ncx, ncz, mode))
    if not os.path.exists(path):
        return None
    total, found = 0.0, set()
    for line in open(path):
        if line.startswith("| `"):
            cells = [c.strip() for c in line.strip().strip("|").split("|")]
            name = cells[0].strip("`")
            if name in kernels and name not in found:
                total += float(cells[-1])
                found.add(name)
    return total if found == set(kernels) else None


def train_surrogate(mdz, hot, m, samples, epochs, batch, lr, seed):
    """Training data from the FP64 reference rheology on the GPU, then Adam
    epochs with the BF16 matrix-core kernels.  Returns (weights, info)."""
    net = C.c_void_p()
    mdz.check(hot.mdz_mlp_create(C.byref(net), C.byref(m.m.materials), C.byref(m.m.model), C.byref(m.m.scaling)))
    try:
        t0 = time.perf_counter()
        mdz.check(hot.mdz_mlp_generate(net, samples, seed))
        t1 = time.perf_counter()
        mdz.check(hot.mdz_mlp_init(net, seed + 1))
        hist = (C.c_double * epochs)()
        mdz.check(hot.mdz_mlp_train(net, epochs, batch, lr, seed + 2, hist))
        t2 = time.perf_counter()
        w = (C.c_float * mdz.MLP_NPARAMS)()
        mdz.check(hot.mdz_mlp_get_weights(net, w, mdz.MLP_NPARAMS))
    finally:
        hot.mdz_mlp_destroy(net)
    info = {"samples": samples, "epochs": epochs, "batch": batch, "lr": lr, "generate_s": round(t1 - t0, 3),
            "train_s": round(t2 - t1, 3), "final_mse": hist[epochs - 1]}
    return w, info


def iteration_stats(mdz, hot, ctx):
    """Mean local iterations of one extra (untimed) unit: FP64, plastic, FP32."""
    mdz.check(hot.mdz_ctx_collect_histogram(ctx, 1))
    mdz.check(hot.mdz_ctx_newton_unit(ctx, None))
    h = (C.c_longlong * 192)()
    mdz.check(hot.mdz_ctx_iteration_histogram(ctx, h))
    mdz.check(hot.mdz_ctx_collect_histogram(ctx, 0))
    out = {}
    for name, a in (("fp64", 0), ("plastic", 64), ("fp32", 128)):
        cnt = sum(h[a:a + 64])
        out[name] = round(sum(i * h[a + i] for i in range(64)) / cnt, 3) if cnt else 0.0
    return out


_HOST = {}


def host_cpu():
    """CPU model, logical CPUs this process may run on, physical cores among
    them, and the OpenMP binding in effect (for the CPU baseline's record).
    Read once, before the OpenMP runtime binds the main thread to one place."""
    if _HOST:
        return dict(_HOST)
    model, phys = "unknown", set()
    cur = {}
    try:
        for line in open("/proc/cpuinfo"):
            if ":" not in line:
                if "processor" in cur:
                    phys.add((cur.get("physical id", "0"), cur.get("core id", cur["processor"]),
                              int(cur["processor"])))
                cur = {}
                continue
            k, v = [x.strip() for x in line.split(":", 1)]
            cur[k] = v
            if k == "model name":
                model = v
    except OSError:
        pass
    allowed = sorted(os.sched_getaffinity(0))
    cores = {(p, c) for p, c, i in phys if i in allowed}
    _HOST.update({"model": model, "cpus_allowed": len(allowed), "physical_cores_allowed": len(cores) or None,
                  "OMP_NUM_THREADS": os.environ.get("OMP_NUM_THREADS"),
                  "OMP_PROC_BIND": os.environ.get("OMP_PROC_BIND", "close"),
                  "OMP_PLACES": os.environ.get("OMP_PLACES", "cores")})
    return dict(_HOST)


def cpu_baseline(mdz, ncx, ncz, seed, units, model_args=()):
    """The oracle (C/OpenMP restatement) on the host cores: full-size units,
    one warm-up then the median of `units`.  Threads bound close, one per
    core (set before the OpenMP runtime starts, when the caller has not)."""
    os.environ.setdefault("OMP_PROC_BIND", "close")
    os.environ.setdefault("OMP_PLACES", "cores")
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_bind

    orc = oracle_bind.load(mdz)
    m = mdz.Model.lithosphere(ncx, ncz, seed, *model_args)
    S = mdz.SparseMat()
    orc.orc_EvalNumberOfEquations(m.m.mesh, C.byref(S))
    blk = [mdz.SparseMat() for _ in range(8)]
    for i, b in enumerate(blk):
        orc.orc_salloc(C.byref(b), S.neq_mom if i % 4 < 2 else S.neq_cont)
    times = []
    for r in range(units + 1):
        t0 = time.perf_counter()
        orc.orc_newton_unit(m.m.mesh, C.byref(m.m.materials), C.byref(m.m.model), C.byref(m.m.Nmodel),
                            C.byref(m.m.scaling), C.byref(S), *[C.byref(b) for b in blk])
        dt = time.perf_counter() - t0
        for b in blk:
            orc.orc_free_block(C.byref(b))
        if r > 0:
            times.append(dt)
    m.free()
    times.sort()
    t = times[len(times) // 2]
    return ncx * ncz / t, orc.orc_num_threads(), t


def marker_step(mdz, hot, ctx, m, per_cell, steps, with_cpu):
    """The device-resident marker-to-grid step (phase fractions at
    centroids and vertices, then cohesion / friction / dilatancy from the
    plastic strain) on per_cell[0] x per_cell[1] seeded markers per cell,
    markers already in HBM: binning (radix sort) and the gathers, host wall
    clock over `steps` calls (each ends with a synchronisation).  Beside it
    the oracle's sequential sums on the same markers, once."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import markers_util

    mk = markers_util.seed_markers(mdz, m, per_cell, seed=7, phase="layers", inactive=0.02)
    t0 = time.perf_counter()
    mdz.check(hot.mdz_ctx_markers_to_grid(ctx, m.m.mesh, C.byref(mk.m), 0))
    first = time.perf_counter() - t0
    mdz.check(hot.mdz_ctx_markers_to_grid(ctx, m.m.mesh, None, 0))
    t0 = time.perf_counter()
    for _ in range(steps):
        mdz.check(hot.mdz_ctx_markers_to_grid(ctx, m.m.mesh, None, 0))
    ms = (time.perf_counter() - t0) / steps * 1e3
    g = m.m.mesh.contents
    nodes = (g.Nx - 1) * (g.Nz - 1) + g.Nx * g.Nz
    # each marker's x, z, phase and plastic strain read once (28 B), three
    # phase fractions and C, friction, dilatancy written per node (48 B)
    alg = mk.n * 28 + nodes * 48
    out = {"markers": mk.n, "per_cell": list(per_cell), "ms": round(ms, 3),
           "markers_per_s": round(mk.n / (ms * 1e-3), 1),
           "algorithmic_bytes": alg, "GBs": round(alg / (ms * 1e-3) / 1e9, 1),
           "frac": round(alg / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
           "first_call_with_upload_ms": round(first * 1e3, 1),
           "note": "not the metric: the per-time-step producers of the rheology's phase fractions and "
                   "strength parameters (P2Mastah, CohesionFrictionDilationGrid), markers resident in HBM"}
    if with_cpu:
        import oracle_bind

        orc = oracle_bind.load(mdz)
        mo = m.clone()
        t0 = time.perf_counter()
        mg = mo.m.mesh.contents
        for centroid, tags in ((1, mg.BCp), (0, mg.BCg)):
            orc.orc_P2Mastah(C.byref(mo.m.model), mk.m, None, mo.m.mesh, None, C.cast(tags.type, C.c_char_p), 0, 0,
                             1, centroid, mo.m.model.itp_stencil)
        orc.orc_CohesionFrictionDilationGrid(mo.m.mesh, C.byref(mk.m), mo.m.materials, mo.m.model, mo.m.scaling)
        out["cpu_oracle_ms"] = round((time.perf_counter() - t0) * 1e3, 1)
        out["cpu_oracle_cores"] = 1
        mo.free()
    return out


def at_abi_ms(mdz, hot, ctx, m, reps):
    """Milliseconds per unit with the host transfers of the drop-in boundary:
    upload of u, v, p, the unit, download of the values and right-hand
    sides of the eight CSR blocks and of the residual vectors (pageable
    host buffers)."""
    import numpy as np

    DP = C.POINTER(C.c_double)
    nu, nw, nc = m.Nx * (m.Nz + 1), (m.Nx + 1) * m.Nz, (m.Nx - 1) * (m.Nz - 1)
    u, v, p = np.zeros(nu), np.zeros(nw), np.zeros(nc)
    mdz.check(hot.mdz_ctx_download_solution(ctx, u.ctypes.data_as(DP), v.ctypes.data_as(DP), p.ctypes.data_as(DP)))
    bufs = []
    for i in range(8):
        neq, nnz = C.c_int(), C.c_int()
        mdz.check(hot.mdz_ctx_block_info(ctx, i, C.byref(neq), C.byref(nnz)))
        bufs.append((np.zeros(max(nnz.value, 1)), np.zeros(max(neq.value, 1))))
    fm, fc = np.zeros(len(bufs[0][1])), np.zeros(len(bufs[3][1]))
    times = []
    for r in range(reps + 1):
        t0 = time.perf_counter()
        mdz.check(hot.mdz_ctx_upload_solution(ctx, u.ctypes.data_as(DP), v.ctypes.data_as(DP), p.ctypes.data_as(DP)))
        mdz.check(hot.mdz_ctx_newton_unit(ctx, None))
        for i, (A, b) in enumerate(bufs):
            mdz.check(hot.mdz_ctx_download_block(ctx, i, None, None, A.ctypes.data_as(DP), b.ctypes.data_as(DP), None))
        mdz.check(hot.mdz_ctx_download_residual(ctx, fm.ctypes.data_as(DP), fc.ctypes.data_as(DP)))
        if r:
            times.append((time.perf_counter() - t0) * 1e3)
    return sum(times) / len(times)


def line_search_ms(mdz, hot, ctx, reps):
    """Milliseconds per call of the five-trial line search (alpha = 0.2 ..
    1.0 of a zero correction, i.e. at the current iterate), host transfers
    of the correction included."""
    import numpy as np

    na, nc = C.c_int(), C.c_int()
    mdz.check(hot.mdz_ctx_block_info(ctx, 0, C.byref(na), None))
    mdz.check(hot.mdz_ctx_block_info(ctx, 3, C.byref(nc), None))
    dx = np.zeros(na.value + nc.value)
    a = np.array([0.2, 0.4, 0.6, 0.8, 1.0])
    out = np.zeros(15)
    DP = C.POINTER(C.c_double)
    args = (ctx, dx.ctypes.data_as(DP), 5, a.ctypes.data_as(DP), out.ctypes.data_as(DP))
    mdz.check(hot.mdz_ctx_line_search(*args))
    t0 = time.perf_counter()
    for _ in range(reps):
        mdz.check(hot.mdz_ctx_line_search(*args))
    return (time.perf_counter() - t0) / reps * 1e3


def device_solve(mdz, hot, ncx, ncz, seed, penalty=1e5):
    """The device solve of the Newton correction (KillerSolver: Powell-Hestenes
    iterations around GCR, preconditioned by the sparse Cholesky factor of the
    penalised Picard operator) on the blocks of one Newton-iteration unit of
    a lithosphere model; the second of two solves is reported (the first
    one also analyses the pattern, allocates the factor and captures the
    preconditioner's launches).  Not the metric."""
    m = mdz.Model.lithosphere(ncx, ncz, seed)
    m.m.model.penalty = penalty
    ctx = C.c_void_p()
    mdz.check(hot.mdz_ctx_create(C.byref(ctx), m.m.mesh, C.byref(m.m.materials), C.byref(m.m.model),
                                 C.byref(m.m.scaling)))
    try:
        mdz.check(hot.mdz_ctx_newton_unit(ctx, None))
        info = mdz.solve_info()
        for _ in range(2):
            t0 = time.perf_counter()
            mdz.check(hot.mdz_ctx_solve(ctx, 0, None, C.byref(info)))
            wall = (time.perf_counter() - t0) * 1e3
        nu, nnz = C.c_int(), C.c_int()
        mdz.check(hot.mdz_ctx_block_info(ctx, 0, C.byref(nu), C.byref(nnz)))
        return {"workload": "lithosphere %dx%d cells, penalty %g, first Newton iteration" % (ncx, ncz, penalty),
                "momentum_unknowns": nu.value, "ms": round(wall, 1), "factor_ms": round(info.factor_ms, 1),
                "iterate_ms": round(info.iterate_ms, 1), "ph_its": info.ph_its,
                "ksp_its": list(info.ksp_its[:info.ph_its]), "kd": info.kd,
                "ms_per_gcr_iteration": round(info.iterate_ms / max(1, info.ksp_its_total), 2)}
    finally:
        hot.mdz_ctx_destroy(ctx)
        m.free()


def ensemble_params(n, seed):
    """Seeded draws of the ensemble: nx U{257..2049} cells, nz = nx / 2,
    friction U[10, 35] deg, cohesion U[5, 50] MPa, extension rate
    log-U[1e-16, 1e-14] 1/s."""
    import numpy as np

    rng = np.random.default_rng(seed)
    out = []
    for i in range(n):
        nx = int(rng.integers(257, 2050))
        out.append((nx, nx // 2, seed * 1000 + i, float(rng.uniform(10.0, 35.0)), float(rng.uniform(5e6, 50e6)),
                    float(10 ** rng.uniform(-16.0, -14.0))))
    return out


def run_ensemble(args, mdz, hot, models=None, steps=None, with_cpu=None):
    """Ensemble of independent lithosphere models, one captured graph launch
    per Newton iteration (every model through one unit), autotuned shapes.
    Returns the bench line of the ensemble workload (a dict)."""
    import numpy as np

    plist = ensemble_params(models or args.models, args.seed)
    steps = steps or args.steps
    with_cpu = (not args.no_cpu) if with_cpu is None else with_cpu
    mode = {"fp64": 0, "mixed": 1, "learned": 2}[args.mode]
    w, training = None, None
    ctxs, cells = [], []
    t0 = time.perf_counter()
    for i, p in enumerate(plist):
        m = mdz.Model.lithosphere(*p)
        if mode == 2 and w is None:
            w, training = train_surrogate(mdz, hot, m, args.train_samples, args.train_epochs, 65536, 1e-3, args.seed)
        c = C.c_void_p()
        mdz.check(hot.mdz_ctx_create(C.byref(c), m.m.mesh, C.byref(m.m.materials), C.byref(m.m.model),
                                     C.byref(m.m.scaling)))
        m.free()
        if w is not None:
            mdz.check(hot.mdz_ctx_set_network(c, w, mdz.MLP_NPARAMS))
        mdz.check(hot.mdz_ctx_set_rheology_mode(c, mode))
        ctxs.append(c)
        cells.append(p[0] * p[1])
        print("model %d/%d: %dx%d ready" % (i + 1, len(plist), p[0], p[1]), file=sys.stderr, flush=True)
    setup_s = time.perf_counter() - t0
    total = sum(cells)
    arr = (C.c_void_p * len(ctxs))(*[c.value for c in ctxs])
    ens = C.c_void_p()
    mdz.check(hot.mdz_ensemble_create(C.byref(ens), arr, len(ctxs)))
    shapes = (C.c_int * (3 * len(ctxs)))()
    br = C.c_int()
    t0 = time.perf_counter()
    mdz.check(hot.mdz_ensemble_autotune(ens, 2, shapes, C.byref(br)))
    tune_s = time.perf_counter() - t0
    print("autotuned: %d chains, %.1f s" % (br.value, tune_s), file=sys.stderr, flush=True)
    for _ in range(args.warmup):
        mdz.check(hot.mdz_ensemble_launch(ens))
    res = np.zeros((len(ctxs), 3))
    mdz.check(hot.mdz_ensemble_residuals(ens, res.ctypes.data_as(C.POINTER(C.c_double))))
    ms = C.c_double()
    mdz.check(hot.mdz_ensemble_time(ens, steps, C.byref(ms)))
    value = total / (ms.value * 1e-3)
    plain_ms, err = None, None
    if mode != 0:
        for c in ctxs:
            mdz.check(hot.mdz_ctx_set_rheology_mode(c, 0))
        pm = C.c_double()
        mdz.check(hot.mdz_ensemble_time(ens, steps, C.byref(pm)))
        plain_ms = pm.value
        ref = np.zeros((len(ctxs), 3))
        mdz.check(hot.mdz_ensemble_residuals(ens, ref.ctypes.data_as(C.POINTER(C.c_double))))
        e = np.abs(res - ref) / np.abs(ref)
        err = {"max": float(e.max()), "median": float(np.median(e.max(axis=1))),
               "per_model_max": [float(x) for x in e.max(axis=1)]}
    sh = np.array(list(shapes)).reshape(-1, 3)
    kinds = {}
    for row in sh:
        k = "%d/%d/%d" % tuple(row)
        kinds[k] = kinds.get(k, 0) + 1
    hot.mdz_ensemble_destroy(ens)
    for c in ctxs:
        hot.mdz_ctx_destroy(c)
    unit_bpc = sum(FUSED_BYTES_PER_CELL.values())  # (the network runs in the rheology kernels' prologue)
    whole = unit_bpc * total / (ms.value * 1e-3) / 1e9

    cpu = None
    if with_cpu:
        # bounded sample: full units of the smallest models of the ensemble
        order = sorted(range(len(plist)), key=lambda i: cells[i])
        done_cells, done_t, used = 0, 0.0, []
        for i in order:
            if done_t > 10.0:
                break
            v, cores, t = cpu_baseline(mdz, plist[i][0], plist[i][1], plist[i][2], 1, model_args=plist[i][3:])
            done_cells += cells[i]
            done_t += t
            used.append(i)
        cpu = {"value": round(done_cells / done_t, 1), "unit": "cell-updates/s", "cores": cores, "kind": "port",
               "sample": "one Newton unit (after 1 warm-up) of each of the %d smallest models of the ensemble, "
                         "%d cells, %.2f s in total" % (len(used), done_cells, done_t), "host": host_cpu()}

    line = {
        "metric": "Newton-iter cell-updates/s (rheol+resid+assembly): learned+FP32 vs plain FP64",
        "value": round(value, 1),
        "unit": "cell-updates/s",
        "n_gpus": 1,
        "steps": steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms.value, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if mode == 0 else "f32+f64",
        "data": "synthetic (seeded lithosphere models)",
        "config": {"workload": "ensemble of %d lithosphere models, nx U{257..2049} x nz = nx/2 cells, friction "
                               "U[10,35] deg, cohesion U[5,50] MPa, rate log-U[1e-16,1e-14] 1/s; one graph launch "
                               "= one Newton-iteration unit of every model" % len(plist),
                   "rheology": args.mode, "models": len(plist), "cells": total, "graph_chains": br.value,
                   "shapes_rheo/picard/jacobian": kinds, "parallelism": "single GPU"},
        "roofline": {"bound": "hbm", "achieved": round(whole, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(whole / HBM_PEAK_GBS, 4), "traffic": None, "stage": "whole unit",
                     "bytes_per_cell": unit_bpc},
        "cpu_baseline": cpu,
        "setup_s": round(setup_s, 1),
        "autotune_s": round(tune_s, 1),
    }
    if plain_ms is not None:
        line["plain_fp64_ms_per_step"] = round(plain_ms, 4)
        line["speedup_vs_plain_fp64"] = round(plain_ms / ms.value, 4)
        line["residual_rel_err_vs_fp64"] = err
    if training is not None:
        line["surrogate_training"] = training
    return line


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--ncx", type=int, default=2049)
    ap.add_argument("--ncz", type=int, default=1025)
    ap.add_argument("--mode", default="learned", choices=["fp64", "mixed", "learned"],
                    help="local iterations: plain FP64, FP32 + FP64 polish, or the network's guess + FP32 + FP64 "
                         "polish (the plain FP64 unit is timed beside the other two)")
    ap.add_argument("--kernel", default="auto", choices=["auto", "generic"],
                    help="grid rheology kernel: log-space where it applies (auto) or the generic one")
    ap.add_argument("--seed", type=int, default=1)
    ap.add_argument("--cpu-units", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--probe-mb", type=int, default=1024, help="size of the HBM copy probe (MiB)")
    ap.add_argument("--train-samples", type=int, default=1 << 24, help="surrogate training samples (learned mode)")
    ap.add_argument("--train-epochs", type=int, default=20)
    ap.add_argument("--workload", default="single", choices=["single", "ensemble"],
                    help="one model of --ncx x --ncz cells, or an ensemble of --models seeded models")
    ap.add_argument("--models", type=int, default=64)
    ap.add_argument("--no-autotune", action="store_true", help="default block shapes instead of autotuned ones")
    ap.add_argument("--no-markers", action="store_true",
                    help="single workload: leave out the marker-to-grid step measured beside it")
    ap.add_argument("--no-solve", action="store_true", help="skip the device solve of the Newton correction")
    ap.add_argument("--no-ensemble", action="store_true",
                    help="single workload: leave out the 64-model ensemble measured beside it")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: the path is built and measured on a single MI355X; "
              "multi-GPU runs are not part of this build (--gpus %d refused)" % args.gpus)
        sys.exit(2)

    host_cpu()
    mdz = _pkg()
    hot = mdz.lib_hot()
    mdz.check(hot.mdz_set_rheology_kernel(0 if args.kernel == "auto" else 1))
    if args.workload == "ensemble":
        print(json.dumps(run_ensemble(args, mdz, hot)))
        return
    m = mdz.Model.lithosphere(args.ncx, args.ncz, args.seed)
    ctx = C.c_void_p()
    mdz.check(hot.mdz_ctx_create(C.byref(ctx), m.m.mesh, C.byref(m.m.materials), C.byref(m.m.model),
                                 C.byref(m.m.scaling)))
    mode = {"fp64": 0, "mixed": 1, "learned": 2}[args.mode]
    training = None
    if mode == 2:
        w, training = train_surrogate(mdz, hot, m, args.train_samples, args.train_epochs, 65536, 1e-3, args.seed)
        mdz.check(hot.mdz_ctx_set_network(ctx, w, mdz.MLP_NPARAMS))
    mdz.check(hot.mdz_ctx_set_rheology_mode(ctx, mode))
    cells = args.ncx * args.ncz
    shape = (C.c_int * 3)()
    if not args.no_autotune:
        # block shapes picked by the autotuner (an ensemble of this one model)
        ens = C.c_void_p()
        mdz.check(hot.mdz_ensemble_create(C.byref(ens), (C.c_void_p * 1)(ctx.value), 1))
        mdz.check(hot.mdz_ensemble_autotune(ens, 5, shape, None))
        hot.mdz_ensemble_destroy(ens)
    mdz.check(hot.mdz_ctx_get_launch_shape(ctx, shape))

    for _ in range(args.warmup):
        mdz.check(hot.mdz_ctx_newton_unit(ctx, None))
    res = (C.c_double * 3)()
    mdz.check(hot.mdz_ctx_newton_unit(ctx, res))
    ms = C.c_double()
    t0 = time.perf_counter()
    mdz.check(hot.mdz_ctx_time_units(ctx, args.steps, C.byref(ms)))
    wall = (time.perf_counter() - t0) / args.steps * 1e3
    ms_per_step = ms.value
    value = cells / (ms_per_step * 1e-3)

    probe = C.c_double()
    mdz.check(hot.mdz_copy_probe(args.probe_mb << 20, 10, C.byref(probe)))

    iters = iteration_stats(mdz, hot, ctx)
    abi_ms = at_abi_ms(mdz, hot, ctx, m, 3)
    ls_ms = line_search_ms(mdz, hot, ctx, 5)
    plain_ms = None
    if mode != 0:
        mdz.check(hot.mdz_ctx_set_rheology_mode(ctx, 0))
        pm = C.c_double()
        mdz.check(hot.mdz_ctx_time_units(ctx, args.steps, C.byref(pm)))
        plain_ms = pm.value
        mdz.check(hot.mdz_ctx_set_rheology_mode(ctx, mode))
    # deferred diagnostics (not the metric's value): units that write only
    # the rheology outputs the unit reads; the other outputs are recomputed
    # once, when the grid is downloaded
    mdz.check(hot.mdz_ctx_defer_diagnostics(ctx, 1))
    dm = C.c_double()
    mdz.check(hot.mdz_ctx_newton_unit(ctx, None))
    mdz.check(hot.mdz_ctx_time_units(ctx, args.steps, C.byref(dm)))
    mdz.check(hot.mdz_ctx_defer_diagnostics(ctx, 0))
    mdz.check(hot.mdz_ctx_newton_unit(ctx, None))
    # learned mode: the separate inference pass (mdz_ctx_fuse_guess(0))
    # instead of the network in the rheology kernels' prologue, timed beside
    separate_ms = None
    if mode == 2:
        mdz.check(hot.mdz_ctx_fuse_guess(ctx, 0))
        fm = C.c_double()
        mdz.check(hot.mdz_ctx_newton_unit(ctx, None))
        mdz.check(hot.mdz_ctx_time_units(ctx, args.steps, C.byref(fm)))
        mdz.check(hot.mdz_ctx_fuse_guess(ctx, 1))
        mdz.check(hot.mdz_ctx_newton_unit(ctx, None))
        separate_ms = fm.value

    st = (C.c_double * 11)()
    mdz.check(hot.mdz_ctx_stage_times(ctx, 3, st))
    stage_ms = {s: st[i] for i, s in enumerate(STAGES)}
    bpc = dict(FUSED_BYTES_PER_CELL)
    # (the network runs in the rheology kernels' prologue: no bytes of its own)
    dom = max(STAGES, key=lambda s: stage_ms[s])
    dom_bytes = bpc[dom] * cells
    achieved = dom_bytes / (stage_ms[dom] * 1e-3) / 1e9
    kern = stage_kernels(tuple(shape), mode == 2)
    per_stage = {}
    for s_ in STAGES:
        if not kern[s_]:
            continue  # a J = 0 stage of the fused D pass: nothing runs
        t = traffic_from_profile(kern[s_], args.ncx, args.ncz, args.mode)
        per_stage[s_] = {"ms": round(stage_ms[s_], 4), "bytes_per_cell": bpc[s_],
                         "GBs": round(bpc[s_] * cells / (stage_ms[s_] * 1e-3) / 1e9, 1),
                         "frac": round(bpc[s_] * cells / (stage_ms[s_] * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
                         "traffic": round(t) if t is not None else None}
    traffic = per_stage[dom]["traffic"]
    roofline = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBS, 4),
                "traffic": round(traffic) if traffic is not None else None,
                "stage": dom, "kernels": kern[dom], "algorithmic_bytes": dom_bytes,
                "bytes_per_cell": bpc[dom], "launch_ms": round(stage_ms[dom], 4),
                "probe_GBs": round(probe.value, 1), "frac_of_probe": round(achieved / probe.value, 4)}
    whole = sum(bpc.values()) * cells / (ms_per_step * 1e-3) / 1e9
    markers = None
    if not args.no_markers:
        markers = marker_step(mdz, hot, ctx, m, (4, 4), 5, not args.no_cpu)
    hot.mdz_ctx_destroy(ctx)
    m.free()

    cpu = None
    if not args.no_cpu:
        v, cores, t = cpu_baseline(mdz, args.ncx, args.ncz, args.seed, args.cpu_units)
        cpu = {"value": round(v, 1), "unit": "cell-updates/s", "cores": cores, "kind": "port",
               "sample": "%d full Newton units of the same %dx%d model (median of %d after 1 warm-up), %.2f s each"
                         % (args.cpu_units, args.ncx, args.ncz, args.cpu_units, t), "host": host_cpu()}

    line = {
        "metric": "Newton-iter cell-updates/s (rheol+resid+assembly): learned+FP32 vs plain FP64",
        "value": round(value, 1),
        "unit": "cell-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if mode == 0 else "f32+f64",
        "data": "synthetic (seeded lithosphere model)",
        "config": {"workload": "lithosphere %dx%d cells, 3 phases VEP, one Newton-iteration unit" % (args.ncx, args.ncz),
                   "rheology": args.mode, "rheology_kernel": args.kernel, "cells": cells,
                   "shape_rheo/picard/jacobian": "%d/%d/%d" % tuple(shape),
                   "parallelism": "single GPU"},
        "roofline": roofline,
        "cpu_baseline": cpu,
        "stages": per_stage,
        "whole_unit_algorithmic_GBs": round(whole, 1),
        "whole_unit_bytes_per_cell": sum(bpc.values()),
        "at_abi_ms_per_step": round(abi_ms, 2),
        "at_abi_value": round(cells / (abi_ms * 1e-3), 1),
        "line_search_5_trials_ms": round(ls_ms, 3),
        "deferred_diagnostics": {"ms_per_unit": round(dm.value, 4),
                                 "ms_per_unit_6_iterations": round((5 * dm.value + ms_per_step) / 6, 4),
                                 "note": "not the metric: the rheology diagnostics are written once per "
                                         "6 Newton iterations (last unit full), as a time step needs them"},
        "host_wall_ms_per_step": round(wall, 4),
        "residual_norms": list(res),
        "local_iterations_mean": iters,
    }
    if plain_ms is not None:
        line["plain_fp64_ms_per_step"] = round(plain_ms, 4)
        line["speedup_vs_plain_fp64"] = round(plain_ms / ms_per_step, 4)
    if separate_ms is not None:
        line["separate_guess_pass_ms_per_step"] = round(separate_ms, 4)
    if training is not None:
        line["surrogate_training"] = training
    if markers is not None:
        line["marker_step"] = markers
    if not args.no_solve:
        line["device_solve"] = device_solve(mdz, hot, 513, 257, args.seed)
    if not args.no_ensemble:
        # the 64-model ensemble workload in the same run (its own line is
        # bench.py --workload ensemble); not the metric's value
        t0 = time.perf_counter()
        ens = run_ensemble(args, mdz, hot, models=args.models, steps=10, with_cpu=False)
        line["ensemble"] = {k: ens.get(k) for k in ("value", "ms_per_step", "plain_fp64_ms_per_step",
                                                     "speedup_vs_plain_fp64", "roofline", "setup_s", "autotune_s")}
        line["ensemble"]["config"] = ens["config"]
        line["ensemble"]["residual_rel_err_vs_fp64_max"] = (ens.get("residual_rel_err_vs_fp64") or {}).get("max")
        line["ensemble"]["wall_s"] = round(time.perf_counter() - t0, 1)
    print(json.dumps(line))


if __name__ == "__main__":
    main()
