"""Benchmark: linear-static solves/s on one MI355X.

Workload (the headline configuration): 1 m x 1 m flat plate, 400 x 400 MITC4
quads (160,801 nodes, 964,806 DOF), thickness 5 mm, E = 70 GPa, nu = 0.3,
simply supported edges, transverse pressure 1 kPa sin(pi x) sin(pi y)
(consistent nodal loads); right-preconditioned GMRES to 1e-8 relative
residual, plain FP64 and mixed precision.

Ordering and fill: the configuration names RCM + ILU(3).  On this thin plate
(t/L = 1/200) the RCM-ordered ILU(3) factors are unstable (negative pivots
of an SPD matrix; |M^-1 b| / |b| ~ 1e6 at 200 x 200) and GMRES stagnates
(the ``configs_as_written`` block records the outcome); natural order +
ILU(3) converges but its triangular sweeps have 2,401 dependency levels.
AMD order with more fill keeps paying at 400 x 400: AMD + ILU(k) solve
steps of 1.95 s at k = 16 (482 iterations, 423 levels), 0.62 s at 56 (63
iterations, 1,215 levels), and, with the AMD tie order updating each reach
in reverse, 0.60 s at 56, 0.54 s at 80 and 0.49 s at 96 (23 iterations,
1,372 levels, 257 ms of numeric factorisation); beyond 96 the
factorisation grows faster than the sweeps shrink (0.52 s at 112, 0.56 s
at 128).  The default run is AMD + ILU(96) + GMRES(500);
``--reorder rcm --lev-fill 3`` runs the configuration as written.

A step is one complete numeric solve of that problem with the mesh and the
symbolic data (pattern, reordering, ILU(k) pattern, element->block map,
element colouring) resident in HBM: Jacobian assembly + boundary conditions
+ copy into the ILU pattern + numeric ILU + GMRES, loads already on the
device.  The JSON line reports the fastest converged precision timed over
all K steps as ``value``; every mode run is listed under ``paths`` (FP64,
FP32 ILU and sweeps inside FP64 GMRES, and GMRES-IR with an FP32 inner
operator, which runs 1 + min(K, 3) steps).

Extra fields: ``roofline`` (the dominant kernel, the sweeps, measured with
HIP events on the library's stream; ``traffic`` is the HBM bytes per launch
measured in this run by two rocprofv3 PMC passes over ``--profile-kernels``
started as child processes (``pmc_traffic`` holds every hot kernel's
figure), else the summary committed in profiles/ for this workload, else
null), ``assembly_roofline`` (the FP64 MFMA Jacobian kernel, with its MFMA
rate and PMC traffic), ``cpu_baseline`` (the oracle
built -O3 -march=native on this host, per stage, one thread and all host
threads, see ``sample``), ``configs_as_written`` (the plate with RCM +
ILU(3) and the 256 x 512 cylinder with ILU(2), bounded), ``served`` (the
served request mix at full size: plain FP64 one request at a time, then
Poisson arrivals at 10x the plain rate through the server with worker
streams and with the batched GMRES engines) and ``latency_ms`` p50/p99 over
the timed steps.  ``--mesh cylinder|wingbox`` runs the other workloads;
``--serve`` runs the served request mix alone (its own JSON line);
``--profile-kernels`` a short run of the hot kernels for rocprofv3.
"""
from __future__ import annotations

import argparse
import ctypes
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0  # MI355X HBM3E
FP64_PEAK_TFLOPS = 78.6  # MI355X dense FP64 (vector and matrix)
# FP64 MFMA flops of the element contraction as implemented: the 21 4x4
# tiles on and above the diagonal of K_e (24 x 24) over k = 36 (9 strains x
# 4 quadrature points), 9 x 21 v_mfma_f64_4x4x4 block products of 128 flops
ASM_FLOPS_PER_ELEM = 21 * 9 * 4 * 4 * 4 * 2  # 24,192

# precision modes of gf_options.precision
PREC_NAMES = {0: "fp64", 1: "mixed", 2: "mixed_pc"}


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--nx", type=int, default=400)
    # other workloads for ad-hoc runs (the JSON line names the workload):
    # cylinder R = 1 m, L = 3 m, nc x 2nc quads, t U[1,8] mm, clamped end,
    # 50 kPa + 10 kN/m; wingbox (seeded, ~489k nodes at --wb-scale 1)
    ap.add_argument("--mesh", default="plate",
                    choices=["plate", "cylinder", "wingbox"])
    ap.add_argument("--cyl-nc", type=int, default=256)
    ap.add_argument("--wb-scale", type=float, default=1.0)
    ap.add_argument("--precision", default="all",
                    choices=["all", "both", "fp64", "mixed", "mixed_pc"])
    ap.add_argument("--reorder", default="amd", choices=["natural", "rcm", "amd"])
    ap.add_argument("--lev-fill", type=int, default=96)
    ap.add_argument("--restart", type=int, default=500)
    ap.add_argument("--max-iters", type=int, default=4000)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-pmc", action="store_true",
                    help="skip the rocprofv3 PMC passes (HBM traffic)")
    # served request mix (separate JSON line; see serve_main)
    ap.add_argument("--serve", action="store_true")
    ap.add_argument("--requests", type=int, default=64)
    ap.add_argument("--slots", type=int, default=16)
    ap.add_argument("--serve-scale", type=float, default=1.0)
    ap.add_argument("--rate", type=float, default=0.0,
                    help="Poisson arrival rate (requests/s); 0: "
                         "--rate-factor times the plain rate")
    # arrivals faster than the server completes them (it runs saturated, so
    # the served rate measures what it delivers, not the arrival rate)
    ap.add_argument("--rate-factor", type=float, default=10.0,
                    help="arrival rate as a multiple of the measured plain "
                         "FP64 rate (0: all requests at t = 0)")
    ap.add_argument("--serve-engine", default="both",
                    choices=["streams", "batched", "both"])
    ap.add_argument("--serve-requests", type=int, default=48,
                    help="requests of the served block of the default run")
    ap.add_argument("--no-serve", action="store_true",
                    help="skip the served block of the default run")
    ap.add_argument("--no-configs", action="store_true",
                    help="skip the configurations-as-written block")
    ap.add_argument("--serve-precision", type=int, default=2)
    # AMD + ILU(64): the cylinders of the mix take 34-64 iterations (ILU(32):
    # 100-129); served 8.0 solves/s against 6.1 with ILU(32), plain FP64
    # one at a time 1.46 against 1.70 solves/s
    ap.add_argument("--serve-lev-fill", type=int, default=64)
    ap.add_argument("--serve-stall", type=int, default=4,
                    help="stall_cycles of the served requests")
    ap.add_argument("--seed", type=int, default=0)
    # short kernel-only run for profilers (rocprofv3 --pmc / --kernel-trace)
    ap.add_argument("--profile-kernels", action="store_true")
    ap.add_argument("--residual-floor", action="store_true",
                    help="after the run, compare the FP64 path's true "
                         "residual with the residual that rounding its "
                         "solution to FP64 causes")
    return ap.parse_args()


class HipEvents:
    """hipEvent timing on an arbitrary stream handle (the library's stream)."""

    def __init__(self):
        self.hip = ctypes.CDLL("libamdhip64.so")
        h = self.hip
        h.hipEventCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
        h.hipEventRecord.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
        h.hipEventSynchronize.argtypes = [ctypes.c_void_p]
        h.hipEventElapsedTime.argtypes = [ctypes.POINTER(ctypes.c_float),
                                          ctypes.c_void_p, ctypes.c_void_p]
        h.hipEventDestroy.argtypes = [ctypes.c_void_p]

    def event(self):
        e = ctypes.c_void_p()
        assert self.hip.hipEventCreate(ctypes.byref(e)) == 0
        return e

    def record(self, e, stream):
        assert self.hip.hipEventRecord(e, stream) == 0

    def elapsed_ms(self, a, b):
        assert self.hip.hipEventSynchronize(b) == 0
        ms = ctypes.c_float()
        assert self.hip.hipEventElapsedTime(ctypes.byref(ms), a, b) == 0
        return ms.value


def pmc_traffic(args, nodes, nnzb_ilu):
    """HBM bytes per sweep launch measured with rocprofv3 PMC counters
    (FETCH_SIZE and WRITE_SIZE in two runs, scaled by the same counters on a
    1 GiB device copy) for this workload, read from the summary committed in
    profiles/; None when no summary matches (nodes and ILU blocks)."""
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles",
                        f"pmc_sweep_plate400_amd_ilu{args.lev_fill}.md")
    if args.mesh != "plate" or not os.path.exists(path):
        return None
    vals = {}
    for line in open(path):
        if line.startswith("traffic_") and ":" in line:
            k, v = line.split(":", 1)
            vals[k.strip()] = float(v.split()[0])
    if (vals.get("traffic_nodes") != nodes or
            vals.get("traffic_nnzb_ilu") != nnzb_ilu):
        return None
    return vals.get("traffic_bytes_per_launch")


def live_pmc_traffic(args):
    """HBM bytes of the hot kernels measured in this run: two rocprofv3 PMC
    passes (FETCH_SIZE, then WRITE_SIZE; one counter a pass) over
    ``--profile-kernels`` of the same workload, run as child processes, each
    counter scaled by what it reads for the 1 GiB device-to-device copy that
    run ends with.  Returns per-launch bytes of the sweeps (mean of L and U),
    the SpMV, one assembly (its colour launches summed) and one numeric
    factorisation (its launches summed), or None when rocprofv3 is missing or
    a pass fails (the caller then falls back to the committed summary)."""
    import csv
    import shutil
    import subprocess
    import tempfile

    exe = shutil.which("rocprofv3")
    if not exe or args.mesh != "plate":
        return None
    env = dict(os.environ, TMPDIR="/tmp")
    per = {}
    with tempfile.TemporaryDirectory(dir="/tmp") as td:
        for ctr in ("FETCH_SIZE", "WRITE_SIZE"):
            out = os.path.join(td, ctr.lower())
            cmd = [exe, "--pmc", ctr, "--output-format", "csv", "-d", out,
                   "-o", "run", "--", sys.executable, "-u",
                   os.path.abspath(__file__), "--profile-kernels",
                   "--nx", str(args.nx), "--reorder", args.reorder,
                   "--lev-fill", str(args.lev_fill)]
            print(f"[bench] live PMC pass {ctr}", file=sys.stderr, flush=True)
            try:
                r = subprocess.run(cmd, cwd="/tmp", env=env, timeout=240,
                                   capture_output=True, text=True)
            except subprocess.TimeoutExpired:
                return None
            files = [os.path.join(dp, f) for dp, _, fs in os.walk(out)
                     for f in fs if f.endswith("counter_collection.csv")]
            if r.returncode != 0 or not files:
                return None
            for row in csv.DictReader(open(files[0])):
                name = row["Kernel_Name"]
                per.setdefault((name, ctr), []).append(
                    float(row["Counter_Value"]))

    def vals(pat, ctr):
        return [v for (n, c), vs in per.items() if c == ctr and pat in n
                for v in vs]

    copy_f, copy_w = vals("copyBuffer", "FETCH_SIZE"), vals("copyBuffer",
                                                          "WRITE_SIZE")
    if not copy_f or not copy_w or max(copy_f) <= 0 or max(copy_w) <= 0:
        return None
    gib = float(1 << 30)
    ff = gib / (max(copy_f) * 1024)  # the copy reads 1 GiB
    wf = gib / (max(copy_w) * 1024)  # and writes 1 GiB

    def bytes_of(pat, launches_per_unit=1):
        f, w = vals(pat, "FETCH_SIZE"), vals(pat, "WRITE_SIZE")
        if not f or not w:
            return None
        units = max(1, len(f) // launches_per_unit)
        return (sum(f) * 1024 * ff + sum(w) * 1024 * wf) / units

    # rows in groups, row by row, or both sweeps of a small system in one
    # launch (half of it each, then)
    def sweep_of(lower):
        small = bytes_of("trsv_small_kernel<double")
        return (bytes_of(f"trsv_group_kernel<double, {lower}")
                or bytes_of(f"trsv_syncfree_kernel<double, {lower}")
                or (small and small / 2))

    lo, up = sweep_of("true"), sweep_of("false")
    nasm = len(vals("jacobian_mfma_kernel<true>", "FETCH_SIZE"))
    return {"sweep_bytes_per_launch": (None if lo is None or up is None
                                       else (lo + up) / 2),
            "sweep_lower": lo, "sweep_upper": up,
            "spmv": bytes_of("spmv_kernel<double>"),
            "assembly": bytes_of("jacobian_mfma_kernel<true>", max(1, nasm)),
            "numeric_ilu": bytes_of("ilu_row_", 1 << 30),
            "calibration": {"fetch_kib_per_gib": max(copy_f),
                            "write_kib_per_gib": max(copy_w)}}


def residual_floor(ctx, p, mesh, x, hip_memcpy):
    """The true relative residual of the FP64 path against what FP64 storage
    of the solution allows: eps |K| |x| (a bound on the residual that
    rounding x causes) and the residual change when every entry of x moves
    by a half unit in the last place with random sign.  A correctly rounded
    solution has a residual of the order of the latter."""
    import torch

    import gpu_fem_amd as G

    L = G.lib()
    d = p.device_arrays()
    nn, nk, _ = p.sizes()
    perm = p.perm()

    def permute(v):
        out = np.empty_like(v)
        out.reshape(-1, 6)[perm] = v.reshape(-1, 6)
        return out

    loads = mesh.loads.copy()
    loads[mesh.bcs] = 0.0
    kv = torch.empty(36 * nk, dtype=torch.float64, device="cuda")
    ctx.sync()
    assert hip_memcpy(ctypes.c_void_p(kv.data_ptr()),
                      ctypes.c_void_p(d["kvals"]), kv.numel() * 8, 3) == 0
    db = torch.from_numpy(permute(loads)).cuda()
    xp = permute(x)
    rowp, cols = ctypes.c_void_p(d["krowp"]), ctypes.c_void_p(d["kcols"])

    def resid(xv):
        dx = torch.from_numpy(xv).cuda()
        r = torch.zeros_like(db)
        ctx.check(L.gf_bsr_resid_comp_f64(ctx.h, nn, rowp, cols, G.ptr(kv),
                                          G.ptr(dx), G.ptr(db), G.ptr(r)))
        ctx.sync()
        return r

    half_ulp = np.finfo(np.float64).eps / 2
    kabs, ax = kv.abs(), torch.from_numpy(np.abs(xp)).cuda()
    y = torch.zeros_like(db)
    ctx.check(L.gf_bsr_spmv_f64(ctx.h, nn, rowp, cols, G.ptr(kabs), G.ptr(ax),
                                G.ptr(y)))
    ctx.sync()
    bn = db.norm().item()
    r0 = resid(xp)
    rng = np.random.default_rng(0)
    r1 = resid(xp * (1.0 + half_ulp * rng.choice([-1.0, 1.0], xp.size)))
    return {"true_rel_resid": r0.norm().item() / bn,
            "eps_absK_absx_over_b": half_ulp * y.norm().item() / bn,
            "half_ulp_random_change": (r1 - r0).norm().item() / bn}


def sweep_bytes(mrp, mcp, w):
    """Algorithmic bytes of one L and one U sweep (values + column indices of
    the triangle incl. the diagonal block, row pointers, rhs read, solution
    written)."""
    n = len(mrp) - 1
    rows = np.repeat(np.arange(n), np.diff(mrp))
    lower = int(np.sum(mcp < rows))
    upper = int(np.sum(mcp > rows))
    blk = 36 * w + 4
    vec = 6 * n * w
    lb = (lower + n) * blk + 8 * (n + 1) + 2 * vec
    ub = (upper + n) * blk + 8 * (n + 1) + 2 * vec
    return lb, ub


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for --gpus "
              f"{args.gpus}); the multi-GPU path is design-only",
              file=sys.stderr)
        sys.exit(2)
    if args.serve:
        # one hardware queue per worker stream (HIP's default is 4), set
        # before the HIP runtime starts
        q = int(os.environ.get("GPU_MAX_HW_QUEUES", "4"))
        if q < min(args.slots, 32):
            os.environ["GPU_MAX_HW_QUEUES"] = str(min(args.slots, 32))
        serve_main(args)
        return
    if args.profile_kernels:
        profile_kernels_main(args)
        return
    if not args.no_serve:
        # the served block's worker streams: one hardware queue each (HIP's
        # default is 4), set before the HIP runtime starts
        q = int(os.environ.get("GPU_MAX_HW_QUEUES", "4"))
        if q < min(args.slots, 32):
            os.environ["GPU_MAX_HW_QUEUES"] = str(min(args.slots, 32))
    import torch

    import gpu_fem_amd as G
    from gpu_fem_amd import meshes as M

    torch.cuda.init()
    nx = args.nx
    t0 = time.time()
    if args.mesh == "cylinder":
        nc = args.cyl_nc
        mesh = M.cylinder(nc, 2 * nc, seed=args.seed)
        wl = (f"cylinder R=1m L=3m {nc}x{2 * nc} MITC4, t U[1,8] mm (seed "
              f"{args.seed}), clamped, 50 kPa + 10 kN/m")
    elif args.mesh == "wingbox":
        f = args.wb_scale
        mesh = M.wingbox(nc=max(2, round(120 * f)), nh=max(2, round(16 * f)),
                         nsb=max(1, round(30 * f)), seed=args.seed)
        wl = (f"wingbox {mesh.name} (seed {args.seed}), panel t U[2,20] mm, "
              f"root clamped, elliptic pressure 20 kPa")
    else:
        mesh = M.plate(nx, nx, 1.0, 1.0, E=70e9, nu=0.3, thick=0.005, bc="ss",
                       load="sine", load_mag=1e3)
        wl = f"plate {nx}x{nx} MITC4, t=5mm, SS, sine pressure"
    print(f"[bench] mesh {mesh.name}: {mesh.nnodes} nodes in "
          f"{time.time()-t0:.1f}s", file=sys.stderr, flush=True)
    ctx = G.Context(0)
    ev = HipEvents()
    stream = ctx.stream
    d_loads = torch.from_numpy(mesh.loads.copy()).cuda()
    d_x = torch.zeros_like(d_loads)
    precs = {"all": [2, 1, 0], "both": [2, 0], "fp64": [0], "mixed": [1],
             "mixed_pc": [2]}[args.precision]
    results = {}
    problems = {}
    for prec in precs:
        name = PREC_NAMES[prec]
        t0 = time.time()
        reorder_id = {"natural": 0, "rcm": 1, "amd": 2}[args.reorder]
        p = G.Problem(ctx, mesh, reorder=reorder_id, lev_fill=args.lev_fill,
                      restart=args.restart, rtol=1e-8,
                      max_iters=args.max_iters, precision=prec)
        problems[name] = p
        print(f"[bench] {name}: symbolic + upload {time.time()-t0:.1f}s",
              file=sys.stderr, flush=True)
        lat = []
        info = None
        # GMRES-IR (mode 1) takes several times the FP64 step on this plate:
        # it runs 1 + min(K, 3) steps and is reported, not the headline
        steps, warmup = ((min(args.steps, 3), 1) if prec == 1
                         else (args.steps, args.warmup))
        for it in range(warmup + steps):
            torch.cuda.synchronize()
            ctx.sync()
            ts = time.perf_counter()
            p.assemble()
            p.factor()
            _, info = p.solve(d_loads, d_x, raise_on_error=False)
            ctx.sync()
            dt = time.perf_counter() - ts
            print(f"[bench] {name} step {it}: {dt*1e3:.1f} ms iters="
                  f"{info.iterations} resid={info.rel_resid:.2e} "
                  f"asm={info.t_assemble*1e3:.2f}ms fac={info.t_factor*1e3:.1f}ms "
                  f"solve={info.t_solve*1e3:.1f}ms status={info.status}",
                  file=sys.stderr, flush=True)
            if it >= warmup:
                lat.append(dt)
        lat = np.array(lat)
        results[name] = dict(
            steps=steps, warmup=warmup,
            converged=bool(info.status == 0 and info.rel_resid <= 1e-8),
            ms_per_step=float(lat.mean() * 1e3),
            solves_per_s=float(1.0 / lat.mean()),
            p50_ms=float(np.percentile(lat, 50) * 1e3),
            p99_ms=float(np.percentile(lat, 99) * 1e3),
            iterations=int(info.iterations), outer=int(info.outer),
            rel_resid=float(info.rel_resid),
            t_assemble_ms=info.t_assemble * 1e3,
            t_factor_ms=info.t_factor * 1e3, t_solve_ms=info.t_solve * 1e3,
            x_host=d_x.cpu().numpy().copy())

    # mixed vs FP64 solution difference: the FP64 path stands in for the FP64
    # oracle at this size (a CPU oracle solve takes several minutes; the FP64
    # path matches the oracle to 1e-8 on the parity meshes)
    for mname in ("mixed", "mixed_pc"):
        if mname in results and "fp64" in results:
            a, b = results[mname]["x_host"], results["fp64"]["x_host"]
            results[mname]["rel_err_vs_fp64_path"] = float(
                np.linalg.norm(a - b) / np.linalg.norm(b))

    # ---- dominant kernel: the triangular sweeps; time them in isolation
    pname = "fp64" if "fp64" in problems else next(iter(problems))
    p = problems[pname]
    d = p.device_arrays()
    nn, nk, nm = p.sizes()
    # host copies of the ILU pattern for the byte count
    from gpu_fem_amd import _i32  # noqa
    rp_k, cp_k = G.node_graph(mesh.conn, mesh.nnodes)
    perm = p.perm()
    krp, kcp = G.pattern_permute(rp_k, cp_k, perm)
    mrp, mcp = G.iluk_symbolic(krp, kcp, args.lev_fill)
    w = 8
    lb, ub = sweep_bytes(mrp, mcp, w)
    ilu_h = p  # the problem owns the ILU; use the public apply on its buffers
    nrep = 20
    tmp = torch.zeros(6 * nn, dtype=torch.float64, device="cuda")
    xo = torch.zeros_like(tmp)
    b = torch.ones_like(tmp)
    ilu = G.Ilu(ctx, mrp, mcp)
    mv = torch.empty(36 * nm, dtype=torch.float64, device="cuda")
    hip_memcpy = ev.hip.hipMemcpy
    hip_memcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t,
                           ctypes.c_int]
    ctx.sync()
    assert hip_memcpy(ctypes.c_void_p(mv.data_ptr()), ctypes.c_void_p(d["mvals"]),
                      mv.numel() * 8, 3) == 0  # factored values of the problem
    ilu.apply(mv, b, tmp, xo)  # warm
    e0, e1 = ev.event(), ev.event()
    ev.record(e0, stream)
    for _ in range(nrep):
        G.lib().gf_bsr_ilu_apply_f64(ilu.h, G.ptr(mv), G.ptr(b), G.ptr(tmp),
                                     G.ptr(xo))
    ev.record(e1, stream)
    pair_ms = ev.elapsed_ms(e0, e1) / nrep
    ctx.check(G.lib().gf_ilu_check(ilu.h))
    sweep_launch_s = pair_ms * 1e-3 / 2
    sweep_bytes_launch = (lb + ub) / 2
    sweep_gbs = sweep_bytes_launch / sweep_launch_s / 1e9
    info_lv = ilu.info()
    sweep_kernel = {"groups": "trsv_group_kernel", "small": "trsv_small_kernel",
                    "levels": "trsv_level_kernel"}.get(
                        ilu.sweep_info()["kind"], "trsv_syncfree_kernel")
    # the FP32 sweeps of the mixed paths, on the FP64 factors rounded to FP32
    # (a sweep's traffic and dependency latency do not depend on the values)
    mv32, b32 = mv.float(), b.float()
    tmp32, xo32 = torch.zeros_like(b32), torch.zeros_like(b32)
    ilu.apply(mv32, b32, tmp32, xo32)  # warm
    ev.record(e0, stream)
    for _ in range(nrep):
        G.lib().gf_bsr_ilu_apply_f32(ilu.h, G.ptr(mv32), G.ptr(b32),
                                     G.ptr(tmp32), G.ptr(xo32))
    ev.record(e1, stream)
    pair32_ms = ev.elapsed_ms(e0, e1) / nrep
    ctx.check(G.lib().gf_ilu_check(ilu.h))
    lb32, ub32 = sweep_bytes(mrp, mcp, 4)
    sweep32_launch_s = pair32_ms * 1e-3 / 2
    sweep32_bytes_launch = (lb32 + ub32) / 2
    sweep32_gbs = sweep32_bytes_launch / sweep32_launch_s / 1e9
    floor = None
    if args.residual_floor and "fp64" in results:
        floor = residual_floor(ctx, problems["fp64"], mesh,
                               results["fp64"]["x_host"], hip_memcpy)
        print(f"[bench] residual floor: {floor}", file=sys.stderr, flush=True)

    # ---- assembly kernels (Jacobian, colour-ordered scatter as in the
    # problem) in isolation
    d_conn = torch.from_numpy(mesh.conn.astype(np.int32)).cuda()
    d_xp = torch.from_numpy(mesh.xpts.copy()).cuda()
    d_dat = torch.from_numpy(mesh.data.copy()).cuda()
    emap = G.elem_ind_map(mesh.conn, krp, kcp, perm)
    d_map = torch.from_numpy(emap).cuda()
    d_perm = torch.from_numpy(perm).cuda()
    d_k = torch.zeros(36 * nk, dtype=torch.float64, device="cuda")
    L = G.lib()
    plan = ctypes.c_void_p()
    ctx.check(L.gf_asm_plan_create(ctx.h, mesh.nelems, mesh.nnodes,
                                   G.ptr(np.ascontiguousarray(mesh.conn, np.int32)),
                                   G.ptr(np.ascontiguousarray(emap, np.int32)),
                                   nk, ctypes.byref(plan)))
    ncolors = L.gf_asm_plan_colors(plan)
    ctx.sync()
    arep = 10
    for rep in range(2):
        ev.record(e0, stream)
        for _ in range(arep):
            ctx.check(L.gf_assemble_jacobian_colored_f64(
                ctx.h, plan, G.ptr(d_conn), G.ptr(d_xp), None, G.ptr(d_dat),
                G.ptr(d_map), G.ptr(d_perm), G.ptr(d_k), None))
        ev.record(e1, stream)
        asm_ms = ev.elapsed_ms(e0, e1) / arep
    L.gf_asm_plan_destroy(plan)
    asm_bytes = 288 * nk + mesh.nelems * (16 + 64 + 56) + mesh.nnodes * (24 + 48 + 48)
    asm_gbs = asm_bytes / (asm_ms * 1e-3) / 1e9

    # ---- HBM traffic of the hot kernels: rocprofv3 PMC passes (children)
    pmc = None if args.no_pmc else live_pmc_traffic(args)

    # ---- CPU baseline: the oracle on the host, bounded sample
    cpu = None
    if not args.no_cpu_baseline:
        kv_host = np.empty(36 * nk)
        ctx.sync()
        assert hip_memcpy(ctypes.c_void_p(kv_host.ctypes.data),
                          ctypes.c_void_p(d["kvals"]), kv_host.nbytes, 2) == 0
        t0 = time.time()
        cpu = cpu_baseline(mesh, perm, kv_host, results[pname]["iterations"],
                           args.restart, args.lev_fill)
        print(f"[bench] cpu baseline {time.time() - t0:.1f}s",
              file=sys.stderr, flush=True)

    # ---- the configurations as written (RCM + ILU(3) plate, ILU(2) cylinder)
    as_written = None
    if not args.no_configs and args.mesh == "plate" and nx == 400:
        as_written = configs_as_written(args, ctx)

    # ---- served request mix (full size): Poisson arrivals at 10x the plain
    # FP64 rate, worker streams and the batched engines
    served = None
    if not args.no_serve:
        served = serve_measure(args, args.serve_requests, 1.0,
                               args.rate_factor, (0, 1))

    best = None
    for name in ("mixed_pc", "mixed", "fp64"):
        if (name in results and results[name]["converged"] and
                results[name]["steps"] == args.steps):
            if best is None or results[name]["solves_per_s"] > results[best]["solves_per_s"]:
                best = name
    if best is None:
        best = pname
    r = results[best]
    line = {
        "metric": "linear-static solves/s, p50/p99 latency @1e-8 resid; "
                  "assembly %HBM roofline",
        "value": r["solves_per_s"] if r["converged"] else 0.0,
        "unit": "solves/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": r["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if best == "fp64" else "f64/f32",
        "precision_modes": {"fp64": "FP64 ILU, sweeps, SpMV, Arnoldi",
                            "mixed": "GMRES-IR: FP32 ILU, sweeps and inner "
                                     "SpMV; FP64 residual, Arnoldi, update",
                            "mixed_pc": "FP32 ILU and sweeps inside FP64 "
                                        "GMRES (FP64 SpMV, Arnoldi)"},
        "data": "synthetic",
        "config": {"workload": f"{wl}; {args.reorder} order + "
                               f"ILU({args.lev_fill}), GMRES({args.restart}) "
                               f"to 1e-8",
                   "nodes": mesh.nnodes, "dof": 6 * mesh.nnodes,
                   "nnzb_K": nk, "nnzb_ILU": nm, "precision": best},
        "latency_ms": {"p50": r["p50_ms"], "p99": r["p99_ms"]},
        "paths": {k: {kk: vv for kk, vv in v.items() if kk != "x_host"}
                  for k, v in results.items()},
        "roofline": {"bound": "hbm",
                     "kernel": f"{sweep_kernel}<double> (L and U)",
                     "achieved": sweep_gbs, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": sweep_gbs / HBM_PEAK_GBS,
                     "traffic": (pmc["sweep_bytes_per_launch"] if pmc
                                 else pmc_traffic(args, nn, nm)),
                     "traffic_source": (
                         "rocprofv3 PMC passes in this run" if pmc else
                         "profiles/pmc_sweep_plate400_amd_ilu"
                         f"{args.lev_fill}.md" if pmc_traffic(args, nn, nm)
                         else None),
                     "bytes_per_launch": sweep_bytes_launch,
                     "launch_us": sweep_launch_s * 1e6,
                     "levels": [info_lv["levels_lower"], info_lv["levels_upper"]]},
        "residual_floor": floor,
        # the dominant kernel of the mixed paths (FP32 factors and vectors)
        "roofline_fp32_sweep": {
            "bound": "hbm", "kernel": f"{sweep_kernel}<float> (L and U)",
            "achieved": sweep32_gbs, "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": sweep32_gbs / HBM_PEAK_GBS,
            "bytes_per_launch": sweep32_bytes_launch,
            "launch_us": sweep32_launch_s * 1e6},
        "assembly_roofline": {"bound": "hbm",
                              "kernel": f"jacobian_mfma_kernel, {ncolors} "
                                        "colour launches",
                              "achieved": asm_gbs, "peak": HBM_PEAK_GBS,
                              "unit": "GB/s", "frac": asm_gbs / HBM_PEAK_GBS,
                              "bytes_per_launch": asm_bytes,
                              "traffic": pmc["assembly"] if pmc else None,
                              "launch_us": asm_ms * 1e3,
                              # FP64 MFMA rate of the element contraction
                              # (upper-triangle 4x4 tiles of K_e, k = 36)
                              "fp64_mfma": {
                                  "flops_per_element": ASM_FLOPS_PER_ELEM,
                                  "achieved_tflops": ASM_FLOPS_PER_ELEM
                                  * mesh.nelems / (asm_ms * 1e-3) / 1e12,
                                  "peak_tflops": FP64_PEAK_TFLOPS,
                                  "frac": ASM_FLOPS_PER_ELEM * mesh.nelems
                                  / (asm_ms * 1e-3) / 1e12 / FP64_PEAK_TFLOPS}},
        "pmc_traffic": pmc,
        "cpu_baseline": cpu,
        "configs_as_written": as_written,
        "served": served,
    }
    print(json.dumps(line), flush=True)


def profile_kernels_main(args):
    """A short run of the hot kernels for profilers: one Jacobian assembly,
    one numeric factorisation, three L+U sweep pairs and three SpMVs of the
    benchmark problem (FP64, --reorder/--lev-fill), and a device copy of
    1 GiB (the calibration kernel for HBM byte counters)."""
    import torch

    import gpu_fem_amd as G
    from gpu_fem_amd import meshes as M

    torch.cuda.init()
    nx = args.nx
    mesh = M.plate(nx, nx, 1.0, 1.0, E=70e9, nu=0.3, thick=0.005, bc="ss",
                   load="sine", load_mag=1e3)
    ctx = G.Context(0)
    reorder_id = {"natural": 0, "rcm": 1, "amd": 2}[args.reorder]
    p = G.Problem(ctx, mesh, reorder=reorder_id, lev_fill=args.lev_fill,
                  precision=0)
    p.assemble()
    p.factor()
    d = p.device_arrays()
    nn, nk, nm = p.sizes()
    L = G.lib()
    n6 = 6 * nn
    b = torch.ones(n6, dtype=torch.float64, device="cuda")
    tmp = torch.zeros_like(b)
    x = torch.zeros_like(b)
    ilu = p.ilu_handle()
    for _ in range(3):
        ctx.check(L.gf_bsr_ilu_apply_f64(ilu, d["mvals"], G.ptr(b), G.ptr(tmp),
                                         G.ptr(x)))
        ctx.check(L.gf_bsr_spmv_f64(ctx.h, nn, d["krowp"], d["kcols"],
                                    d["kvals"], G.ptr(b), G.ptr(x)))
    ctx.sync()
    src = torch.ones(1 << 27, dtype=torch.float64, device="cuda")  # 1 GiB
    dst = torch.empty_like(src)
    dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"profile_kernels": True, "nodes": nn, "nnzb_K": nk,
                      "nnzb_ILU": nm, "copy_bytes": 2 * src.numel() * 8}),
          flush=True)


SERVE_METRIC = "served linear-static solves/s, p50/p99 latency @1e-8 resid"


def serve_measure(args, nreq, scale, rate_factor, batch_modes):
    """Served request mix: seeded plates and cylinders of differing sizes
    (gpu_fem_amd.meshes.served_requests), each a complete linear-static solve
    to 1e-8 relative residual (symbolic phase, upload, assembly, ILU, GMRES).

    Plain path: FP64, one request at a time on one context.  Served path:
    gf_server with ``--slots`` workers under a 200 GB admission budget, FP32
    ILU and sweeps inside FP64 GMRES (``--serve-precision``), requests
    submitted at Poisson arrival times: rate ``args.rate`` if set, else
    ``rate_factor`` times the measured plain rate (0: all at once, which
    measures capacity).  ``batch_modes``: 0 = each worker solves on its own
    stream, 1 = the batched GMRES engines.  Only requests that end at or
    below the tolerance count as solves; each served result is compared with
    the plain FP64 result of the same request."""
    import gpu_fem_amd as G
    from gpu_fem_amd import meshes as M

    t0 = time.time()
    reqs = M.served_requests(nreq, seed=args.seed, scale=scale)
    print(f"[serve] {len(reqs)} requests generated in {time.time()-t0:.1f}s; "
          f"nodes {min(m.nnodes for m in reqs)}..{max(m.nnodes for m in reqs)}",
          file=sys.stderr, flush=True)
    # AMD + ILU(64) by default (--serve-lev-fill): AMD + ILU(3) stagnates
    # near a relative residual of 1 on the thinner plates and cylinders of
    # this mix, ILU(12) needs re-runs with more fill for the thinnest
    # cylinders, ILU(32) takes 100-129 iterations on the larger cylinders.
    # stall_cycles: a solve whose residual falls by less than 10% over
    # --serve-stall restart cycles stops early (and is re-run with twice the
    # level of fill when it stopped far from the tolerance)
    opts = dict(reorder=2, lev_fill=args.serve_lev_fill, restart=200,
                rtol=1e-8, max_iters=20000, stall_cycles=args.serve_stall)
    ctx = G.Context(0)
    # plain FP64, one at a time
    plain_x, plain_lat, plain_ok = {}, [], 0
    t0 = time.perf_counter()
    plain_escalated = 0
    for i, m in enumerate(reqs):
        ts = time.perf_counter()
        # the server's policy: a solve that ends far from the tolerance (or
        # an ILU or GMRES that breaks down) runs again with twice the level
        # of fill, at most twice
        o = dict(opts)
        for attempt in range(3):
            p = G.Problem(ctx, m, precision=0, **o)
            try:
                p.assemble()
                p.factor()
                x, info = p.solve(raise_on_error=False)
            except G.GfError as e:
                x, info = None, G.SolveInfo()
                info.status = e.code
            p.close()
            far = info.status == -6 and not (info.rel_resid <= 1e3 * o["rtol"])
            if (not (far or info.status in (-4, -5)) or attempt == 2 or
                    o["lev_fill"] >= 64):
                break
            o["lev_fill"] = min(2 * max(o["lev_fill"], 1), 64)
            plain_escalated += 1
        dt = time.perf_counter() - ts
        plain_lat.append(dt)
        plain_ok += int(info.status == 0)
        plain_x[i] = x
        print(f"[serve] plain {i} {m.name}: {dt*1e3:.1f} ms iters="
              f"{info.iterations} resid={info.rel_resid:.2e} status={info.status}",
              file=sys.stderr, flush=True)
    t_plain = time.perf_counter() - t0
    ctx.close()
    plain_sps = plain_ok / t_plain
    rate = args.rate if args.rate > 0 else rate_factor * plain_sps
    rng = np.random.default_rng(args.seed + 1)
    n = len(reqs)
    arrivals = (np.cumsum(rng.exponential(1.0 / rate, n)) if rate > 0
                else np.zeros(n))
    out = {"requests": n, "scale": scale, "seed": args.seed,
           "slots": args.slots, "budget_gb": 200.0,
           "arrival_rate_per_s": rate,
           "arrivals": ("Poisson, rate %.3g/s = %g x the plain rate" %
                        (rate, rate_factor)) if args.rate <= 0 and rate > 0
                       else ("Poisson, rate %.3g/s" % rate if rate > 0
                             else "all at t = 0"),
           "order": "AMD", "lev_fill": args.serve_lev_fill,
           "precision": PREC_NAMES[args.serve_precision], "rtol": 1e-8,
           "plain_fp64_one_at_a_time": {
               "solves_per_s": plain_sps, "ok": plain_ok,
               "p50_ms": float(np.percentile(plain_lat, 50) * 1e3),
               "p99_ms": float(np.percentile(plain_lat, 99) * 1e3),
               "escalated": plain_escalated}}
    for batch in batch_modes:
        os.environ["GPUFEM_SERVE_BATCH"] = str(batch)
        srv = G.Server(budget_gb=200.0, slots=args.slots)
        got = {}

        def drain_ready():
            while True:
                r = srv.poll()
                if r is None:
                    return
                got[r[0]] = r

        t0 = time.perf_counter()
        for i, m in enumerate(reqs):
            while time.perf_counter() - t0 < arrivals[i]:
                drain_ready()
                time.sleep(0.0005)
            code = srv.submit(i, m, precision=args.serve_precision, **opts)
            if code != 0:
                raise RuntimeError(f"submit {i} refused: {code}")
        srv.drain()
        t_served = time.perf_counter() - t0
        drain_ready()
        st = srv.stats()
        srv.close()
        lat = np.array([got[i][3] for i in sorted(got)])
        ok = sum(int(got[i][2].status == 0 and got[i][2].rel_resid <= 1e-8)
                 for i in got)
        errs = []
        for i in sorted(got):
            xs, xp = got[i][1], plain_x[i]
            if xp is None or got[i][2].status != 0:
                continue
            errs.append(float(np.linalg.norm(xs - xp) /
                              max(np.linalg.norm(xp), 1e-300)))
        served_sps = ok / t_served
        name = "served" if batch == 0 else "served_batched"
        out[name] = {
            "engine": ("worker streams" if batch == 0 else
                       "batched GMRES engines (fused launches, HIP graph)"),
            "solves_per_s": served_sps, "ok": ok,
            "failed": {str(i): int(got[i][2].status) for i in sorted(got)
                       if got[i][2].status != 0},
            "makespan_s": t_served,
            "p50_ms": float(np.percentile(lat, 50) * 1e3),
            "p99_ms": float(np.percentile(lat, 99) * 1e3),
            "speedup_vs_plain": served_sps / plain_sps,
            "escalated": int(st.get("escalated", 0)),
            "max_rel_diff_vs_plain_fp64": max(errs) if errs else None,
            "peak_admitted_gb": st["peak_bytes"] / 1e9}
        print(f"[serve] {name}: {served_sps:.2f} solves/s, ok {ok}/{n}, "
              f"{served_sps / plain_sps:.2f}x plain", file=sys.stderr,
              flush=True)
    os.environ.pop("GPUFEM_SERVE_BATCH", None)
    return out


def serve_main(args):
    """--serve: the served mix alone, its own JSON line."""
    import torch

    torch.cuda.init()
    modes = {"streams": (0,), "batched": (1,), "both": (0, 1)}[args.serve_engine]
    r = serve_measure(args, args.requests, args.serve_scale, args.rate_factor,
                      modes)
    key = "served" if "served" in r else "served_batched"
    line = {"metric": SERVE_METRIC, "value": r[key]["solves_per_s"],
            "unit": "solves/s", "n_gpus": 1, "higher_is_better": True,
            "data": "synthetic",
            "config": {"workload": "served request mix: plates n^2, n "
                                   "log-uniform [32, 256], and cylinders "
                                   "64x128..192x384, t U[1,10] mm, p U[0.5,5] "
                                   "kPa, clamped/SS"},
            "latency_ms": {"p50": r[key]["p50_ms"], "p99": r[key]["p99_ms"]},
            "served": r}
    print(json.dumps(line), flush=True)


def configs_as_written(args, ctx):
    """The workloads' own orderings and fills, which do not converge at full
    size: the 400 x 400 plate with RCM + ILU(3) and the 256 x 512 cylinder
    with AMD + ILU(2), each bounded by an iteration limit (and a stall
    window for the plate) so that the outcome is recorded in seconds."""
    import gpu_fem_amd as G
    from gpu_fem_amd import meshes as M

    out = {}
    cases = [
        ("plate400_rcm_ilu3",
         lambda: M.plate(400, 400, 1.0, 1.0, E=70e9, nu=0.3, thick=0.005,
                         bc="ss", load="sine", load_mag=1e3),
         dict(reorder=1, lev_fill=3, restart=500, max_iters=1500,
              stall_cycles=2)),
        ("cylinder256x512_amd_ilu2",
         lambda: M.cylinder(256, 512, seed=args.seed),
         dict(reorder=2, lev_fill=2, restart=500, max_iters=2000,
              stall_cycles=0)),
    ]
    for name, mk, o in cases:
        t0 = time.perf_counter()
        mesh = mk()
        p = G.Problem(ctx, mesh, rtol=1e-8, precision=0, **o)
        try:
            p.assemble()
            p.factor()
            _, info = p.solve(raise_on_error=False)
            res = {"status": int(info.status), "iterations": int(info.iterations),
                   "rel_resid": float(info.rel_resid),
                   "converged": bool(info.status == 0),
                   "limits": o, "wall_s": time.perf_counter() - t0}
        except G.GfError as e:
            res = {"status": int(e.code), "error": str(e), "limits": o,
                   "wall_s": time.perf_counter() - t0}
        p.close()
        out[name] = res
        print(f"[bench] as written {name}: {res}", file=sys.stderr, flush=True)
    return out


def _lscpu():
    """CPU model and logical CPU count of this host (lscpu)."""
    import subprocess

    model, cpus = None, os.cpu_count()
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True,
                             timeout=20).stdout
        for line in out.splitlines():
            k, _, v = line.partition(":")
            if k.strip() == "Model name":
                model = v.strip()
            elif k.strip() == "CPU(s)":
                cpus = int(v.strip())
    except Exception:  # noqa: BLE001 - lscpu missing: report what Python sees
        pass
    return model, cpus


def cpu_baseline(mesh, perm, kv, gpu_iters, restart, lev_fill, reps=5):
    """The reference host path restated by the oracle, built -O3
    -march=native on this host, timed stage by stage on a bounded sample of
    the benchmark problem: the median of ``reps`` runs per stage, with one
    thread and with all host threads this process may use (OMP_NUM_THREADS
    or the CPU count).  Stages: Jacobian assembly (element loop of
    include/base/elem_group.h:121-181, the first 1/50 of the elements, scaled
    to all), symbolic phase (node graph, the product's AMD permutation, the
    permuted pattern, ILU(k) symbolic, element->block map, transpose map; the
    whole problem, sequential), numeric ILU (the leading rows holding 1/100
    of the block updates, scaled by the update count; sequential) and GMRES
    (two iterations of the restart length used on the GPU: ILU sweeps, SpMV,
    modified Gram-Schmidt; scaled to the GPU's iteration count).  One solve
    is assembly + numeric ILU + GMRES, as the GPU step."""
    import statistics
    import tempfile

    import oracle

    model, ncpu = _lscpu()
    nall = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or ncpu or 1
    path = oracle.build_native(os.path.join(tempfile.gettempdir(),
                                            "gpufem_oracle_native"))
    oracle.use_library(path)
    L = oracle.lib()

    def med(fn):
        ts = []
        for _ in range(reps):
            t0 = time.perf_counter()
            fn()
            ts.append(time.perf_counter() - t0)
        return statistics.median(ts)

    n, ne = mesh.nnodes, mesh.nelems
    # symbolic phase (sequential), the whole problem
    def symbolic():
        rp, cp = oracle.node_graph(mesh.conn, n)
        krp, kcp = oracle.permute_pattern(rp, cp, perm)
        mrp, mcp, _ = oracle.iluk(krp, kcp, lev_fill)
        oracle.elem_ind_map(mesh.conn, krp, kcp, perm)
        oracle.transpose(krp, kcp)
        return krp, kcp, mrp, mcp
    krp, kcp, mrp, mcp = symbolic()
    t_sym = med(symbolic)
    emap = oracle.elem_ind_map(mesh.conn, krp, kcp, perm)
    ns = max(1, ne // 50)
    # numeric ILU sample: the first rows holding 1/100 of the block updates
    row_of = np.repeat(np.arange(n), np.diff(mrp))
    dpos = np.flatnonzero(mcp == row_of)
    ulen = mrp[1:] - dpos - 1
    low = mcp < row_of
    upd = np.bincount(row_of[low], weights=ulen[mcp[low]] + 1.0, minlength=n)
    cum = np.cumsum(upd)
    nr = n if cum[-1] <= 0 else int(np.searchsorted(cum, 0.01 * cum[-1])) + 1
    ilu_scale = cum[-1] / cum[nr - 1] if cum[nr - 1] > 0 else 1.0
    mv = oracle.copy_values(krp, kcp, kv, mrp, mcp)
    # the GMRES leg runs on the sample's partly factored values (rows past
    # the sample hold the matrix values): a sweep's and an SpMV's time does
    # not depend on the values, and two iterations need not converge
    lu, _ = oracle.bsr_ilu(mrp, mcp, mv, rows=nr)
    b = oracle.permute_vec(perm, oracle.apply_bcs_vec(mesh.bcs, mesh.loads))
    its = 2
    legs = {}
    for name, nt in (("single_thread", 1), ("all_cores", nall)):
        L.orc_set_threads(nt)
        t_asm = med(lambda: oracle.assemble_jacobian(
            mesh.conn[:ns], mesh.xpts, mesh.data[:ns], emap[:16 * ns], perm,
            int(krp[-1]), with_res=False)) * ne / ns
        t_ilu = med(lambda: oracle.bsr_ilu(mrp, mcp, mv, rows=nr)) * ilu_scale
        t_it = med(lambda: oracle.gmres(krp, kcp, kv, mrp, mcp, lu, b,
                                        restart=restart, max_iters=its,
                                        rtol=1e-30)) / its
        t_solve = t_asm + t_ilu + t_it * max(gpu_iters, 1)
        legs[name] = {"threads": nt, "assembly_s": t_asm, "symbolic_s": t_sym,
                      "numeric_ilu_s": t_ilu, "gmres_iteration_s": t_it,
                      "gmres_s": t_it * max(gpu_iters, 1),
                      "solve_s": t_solve, "solves_per_s": 1.0 / t_solve}
    L.orc_set_threads(1)
    best = legs["all_cores"]
    return {"value": best["solves_per_s"], "unit": "solves/s",
            "cores": nall, "kind": "port",
            "cpu_model": model, "host_cpus": ncpu,
            "build": "oracle, g++ -O3 -march=native -fopenmp (no fast-math)",
            "sample": f"median of {reps} runs per stage: assembly of {ns} of "
                      f"{ne} elements scaled x{ne / ns:.0f}; symbolic phase of "
                      f"the whole problem; numeric ILU of the first {nr} of "
                      f"{n} rows (1/100 of its block updates) scaled "
                      f"x{ilu_scale:.0f}; {its} GMRES iterations scaled to "
                      f"the GPU's {gpu_iters}; one solve = assembly + numeric "
                      f"ILU + GMRES (the GPU step); ILU, sweeps and the "
                      f"symbolic phase are sequential in both legs",
            "legs": legs}


if __name__ == "__main__":
    main()
