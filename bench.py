#!/usr/bin/env python3
"""Benchmark: batched per-Fourier-mode Helmholtz solve and DNS step on one
MI355X.

Helmholtz workload: 16x16 quadrilateral elements on [0,2pi]x[-1,1], N_P=10,
N_Z=64 planes = 32 Fourier modes (beta=1), lambda2=1 so mode k solves with
1+k^2; u=0 on y=+-1, periodic in x; seeded Gaussian forcing with amplitude
(1+k)^-2 per mode.  One step = one Field::solve of all 63 planes (32
mode-solves: mode 0 real, modes 1..31 Re+Im; the Nyquist plane is not
solved), inputs resident in HBM.  Run as the FP64 path and as the mixed
path (FP32 elemental work, FP64 band solve, FP64 residual refinement).

DNS workload: forced periodic channel, 12x24 elements on [0,4pi]x[-1,1],
N_P=8, N_Z=128 (Lz=2pi), Re=2000, dt=1e-3, second-order stiffly-stable
splitting with skew-symmetric advection, Poiseuille + seeded 1e-2
perturbation; 100 steps timed.

Prints ONE JSON line: the Helmholtz rate as `value`, both precision
variants, the DNS rate, a roofline entry for the condensed FP64 solve (the
dissection's levels) measured with HIP events on the solve stream, and the CPU oracle timed on bounded samples of the same
workloads.
"""
from __future__ import annotations

import argparse
import ctypes as C
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "mode-solves/s at ≤1e-10 rel err (mixed vs FP64 GPU); DNS steps/s"
HBM_PEAK_GBS = 8000.0


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=50)
    p.add_argument("--warmup", type=int, default=5)
    p.add_argument("--cpu-seconds", type=float, default=10.0,
                   help="bounded CPU-baseline sample length")
    p.add_argument("--no-cpu-baseline", action="store_true")
    p.add_argument("--no-parity", action="store_true")
    p.add_argument("--dns-steps", type=int, default=100)
    p.add_argument("--dns-warmup", type=int, default=3)
    p.add_argument("--no-dns", action="store_true")
    p.add_argument("--dns-only", action="store_true",
                   help="run only the DNS leg (for kernel profiles)")
    p.add_argument("--no-batch", action="store_true")
    p.add_argument("--no-dealias", action="store_true")
    p.add_argument("--batch-runs", type=int, default=20)
    p.add_argument("--no-mixed", action="store_true")
    p.add_argument("--no-adjoint", action="store_true")
    p.add_argument("--mixed-tol", type=float, default=1e-6,
                   help="relative correction size that ends the mixed refinement (each "
                        "pass contracts the error by ~1e-7, so the pass that applies a "
                        "correction below 1e-6 leaves ~1e-13; the error against the FP64 "
                        "path is measured and reported)")
    p.add_argument("--cpu-dns-child", action="store_true", help=argparse.SUPPRESS)
    p.add_argument("--copy-calibration", action="store_true",
                   help="only copy 256 MiB device to device 3 times (the reference "
                        "kernel for scaling rocprofv3 FETCH_SIZE / WRITE_SIZE)")
    return p.parse_args()


def copy_calibration(torch):
    n = 1 << 28
    a = torch.ones(n, dtype=torch.uint8, device="cuda")
    b = torch.empty_like(a)
    for _ in range(3):
        b.copy_(a)
    torch.cuda.synchronize()
    print(json.dumps({"copy_calibration_bytes": n, "copies": 3}), flush=True)


def cpu_baseline(P, seconds):
    """The CPU oracle (a plain-C FP64 port of the reference's solve) on one
    core: Field::solve of modes 0..7 of the same workload, repeated until
    `seconds` of solve time; set-up (factorisation) excluded."""
    from oracle import oracle as O
    m = P["mesh"]
    n = m.nel * m.npnp
    om = O.OracleMesh(m)
    modes = list(range(8))
    systems = {md: O.OracleMsys(om, P["lambda2"], (P["beta"] * md) ** 2) for md in modes}
    planes = [(0, 0)] + [(md, 2 * md + r) for md in modes[1:] for r in (0, 1)]
    F = P["forcing"]
    t0 = time.perf_counter()
    count = 0
    reps = 0
    while True:
        for md, k in planes:
            systems[md].solve_plane(F[k, :n])
        count += len(modes)
        reps += 1
        el = time.perf_counter() - t0
        if el >= seconds:
            break
    return {"value": count / el, "unit": "mode-solves/s", "cores": 1, "kind": "port",
            "sample": f"oracle Field::solve (plain C, no BLAS), modes 0-7 (15 planes) x {reps} "
                      f"repetitions, {el:.1f} s, same mesh/numbering/forcing, 1 thread; "
                      f"CPU {cpu_model()}"}


THREAD_CAPS = {"OMP_NUM_THREADS": "1", "OPENBLAS_NUM_THREADS": "1", "MKL_NUM_THREADS": "1"}


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline_dns_child(steps=3, timed_from=1):
    """Child-process body (numpy with one BLAS/OpenMP thread): the DNS oracle
    on the full channel workload; systems factorised first and excluded,
    step 1 (first-order start) untimed, steps 2..`steps` timed."""
    from oracle.dns_oracle import DnsOracle
    from semtex_amd.problems import dns_channel
    P = dns_channel()
    O = DnsOracle(P["mesh_u"], P["mesh_p"], P["nz"], P["beta"], P["kinvis"], P["dt"],
                  const_force=P["const_force"], advection="skew")
    t_setup = time.perf_counter()
    for md in range(P["nz"] // 2):
        O.system("p", 0.0, md)
        for q in (1, 2):
            O.system("u", {1: 1.0, 2: 1.5}[q] / (P["dt"] * P["kinvis"]), md)
    t_setup = time.perf_counter() - t_setup
    O.set_initial(P["u0"])
    t_steps = []
    for _ in range(steps):
        t0 = time.perf_counter()
        O.step()
        t_steps.append(time.perf_counter() - t0)
    el = sum(t_steps[timed_from:])
    nt = steps - timed_from
    print(json.dumps({"value": nt / el, "unit": "DNS steps/s", "cores": 1, "kind": "port",
                      "sample": f"DNS oracle (numpy + C solve, one BLAS/OpenMP thread), full "
                                f"channel workload, steps {timed_from + 1}-{steps} timed "
                                f"({el:.1f} s); {3 * P['nz'] // 2} mode systems factorised "
                                f"first ({t_setup:.1f} s, excluded); CPU {cpu_model()}"}),
          flush=True)


def cpu_baseline_dns():
    """The DNS CPU baseline in a child process with every BLAS / OpenMP
    thread pool capped at one thread (the parent has torch and the GPU)."""
    import subprocess
    env = dict(os.environ, **THREAD_CAPS)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), "--cpu-dns-child"],
                       capture_output=True, text=True, env=env, timeout=600)
    if r.returncode != 0:
        raise RuntimeError("DNS CPU baseline failed:\n" + r.stderr[-2000:])
    return json.loads(r.stdout.strip().splitlines()[-1])


def helmholtz_leg(a, P, gm, precision, L, _lib, torch):
    """Set up the modal systems, warm up, time `steps` solves; returns the
    rate, the last solution and per-phase times (FP64 path only)."""
    from semtex_amd.solver import SX_MIXED, Field, ModalMatrixSys
    m, nz, nmodes = P["mesh"], P["nz"], P["nmodes"]
    t0 = time.perf_counter()
    M = ModalMatrixSys(P["lambda2"], P["beta"], 0, nmodes, gm, precision)
    torch.cuda.synchronize()
    setup_s = time.perf_counter() - t0
    F_src = torch.from_numpy(P["forcing"]).cuda()
    u = Field(gm, nz)
    fs = [F_src.clone() for _ in range(a.warmup + a.steps)]
    torch.cuda.synchronize()
    kw = dict(mixed_tol=a.mixed_tol, max_iter=20) if precision == SX_MIXED else {}
    for i in range(a.warmup):
        u.solve(fs[i], M, **kw)
    torch.cuda.synchronize()
    sol = u.data.clone()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t_wall = time.perf_counter()
    e0.record()
    for i in range(a.steps):
        u.solve(fs[a.warmup + i], M, **kw)
    e1.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t_wall
    ms = e0.elapsed_time(e1)
    res = {"M": M, "u": u, "solution": sol, "ms_per_step": ms / a.steps,
           "value": nmodes * a.steps / (ms / 1e3), "setup_s": setup_s, "wall_s": wall,
           "iters": getattr(u, "last_iters", None)}
    if precision != SX_MIXED:
        fs_t = [F_src.clone() for _ in range(a.steps)]
        torch.cuda.synchronize()
        L.sx_timing_enable(1)
        for i in range(a.steps):
            u.solve(fs_t[i], M)
        torch.cuda.synchronize()
        pm = (C.c_double * _lib.SX_NPHASE)()
        pc = (C.c_int * _lib.SX_NPHASE)()
        _lib.check(L.sx_timing_read(pm, pc, _lib.SX_NPHASE), "sx_timing_read")
        L.sx_timing_enable(0)
        res["phases"] = {name: pm[i] / max(pc[i], 1) for i, name in enumerate(_lib.PHASES)}
    return res


def dns_leg(a, torch, dealias=False):
    """DNS channel: set-up, `dns_warmup` untimed steps, `dns_steps` timed
    steps from the same initial field (3/2-rule dealiased products when
    `dealias`)."""
    from semtex_amd.problems import dns_channel
    from semtex_amd.solver import DNS, SX_SKEW, GpuMesh
    P = dns_channel()
    mu = P["mesh_u"]
    n = mu.nel * mu.npnp
    print(f"# DNS mesh {mu.info['nx']}x{mu.info['ny']} np={mu.np} nz={P['nz']} "
          f"nband u/p {mu.nband}/{P['mesh_p'].nband}", file=sys.stderr, flush=True)
    t0 = time.perf_counter()
    gu, gp = GpuMesh(mu), GpuMesh(P["mesh_p"])
    D = DNS(gu, gp, P["nz"], P["beta"], P["kinvis"], P["dt"], const_force=P["const_force"],
            advection=SX_SKEW)
    if dealias:
        D.set_dealias(True)
    u0 = torch.zeros((3, P["nz"], D.stride), dtype=torch.float64)
    u0[:, :, :n] = torch.from_numpy(P["u0"])
    u0 = u0.cuda()
    torch.cuda.synchronize()
    setup_s = time.perf_counter() - t0
    D.set_state(u0)
    D.step(a.dns_warmup)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    D.step(a.dns_steps)
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1)
    ok = all(bool(torch.isfinite(D.field(i)).all()) for i in range(4))
    return {"P": P, "D": D, "u0": u0, "ms_per_step": ms / max(a.dns_steps, 1),
            "value": a.dns_steps / (ms / 1e3), "setup_s": setup_s, "finite": ok}


FIXTURE = os.path.join(ROOT, "tests", "golden", "dns_channel_12x24_np8_nz128.npz")
FIELDS = ("u", "v", "w", "p")


def dns_roofline(dn):
    """Algorithmic HBM bytes of one DNS step over its time: every mode's
    velocity and pressure solve operators read once (the grouped velocity
    solve reads the velocity's once for u, v, w), plus 40 passes over an
    [nz][S] field: advection 6 (u in, N out), waveProp 15 (4 history levels
    of 3 fields in, H out), divergence 4, pressure solve 2, projection 7,
    velocity solves 6."""
    from semtex_amd.solver import ModalMatrixSys
    P, D = dn["P"], dn["D"]
    nm = P["nz"] // 2
    lam2 = 1.5 / (P["dt"] * P["kinvis"])
    band = 8 * nm * sum(ModalMatrixSys(lam, P["beta"], 0, nm, g).layout()["operators"]
                        for lam, g in ((lam2, D.gu), (0.0, D.gp)))
    fields = 40 * 8 * P["nz"] * D.stride
    total = band + fields
    achieved = total / (dn["ms_per_step"] * 1e-3) / 1e9
    return {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4), "algorithmic_bytes": total,
            "operator_bytes": band, "field_bytes": fields}


def dns_parity(dn, torch):
    """Per-step parity of the GPU DNS with the oracle, the measures of
    tests/test_gpu_dns_channel_full.py: (1) steps 1-2 against the oracle
    run here, every Fourier plane (Nyquist excluded), relative L2 per field,
    beside the floor the fixture records for that step (the oracle against
    an independently ordered FP64 solve of the singular mode-0 pressure,
    condition ~2.6e5); (2) steps 1-100 against the committed oracle fixture
    at 256 sampled (plane, node) positions: the velocity components'
    max |error| over the velocity scale (max |u, v, w|), the pressure's over
    max |p| beside 10x the running floor."""
    from oracle.dns_oracle import DnsOracle
    P, D = dn["P"], dn["D"]
    mu, nz = P["mesh_u"], P["nz"]
    n = mu.nel * mu.npnp
    pl = [k for k in range(nz) if k != 1]
    out = {}
    F = np.load(FIXTURE) if os.path.exists(FIXTURE) else None
    O = DnsOracle(mu, P["mesh_p"], nz, P["beta"], P["kinvis"], P["dt"],
                  const_force=P["const_force"], advection="skew")
    O.set_initial(P["u0"])
    D.set_state(dn["u0"])
    live = {f: [] for f in FIELDS}
    for s in range(2):
        O.step()
        D.step(1)
        for i, f in enumerate(FIELDS):
            g = D.field(i).cpu().numpy()[pl, :n]
            o = (O.u[i] if i < 3 else O.p)[pl]
            live[f].append(float(np.linalg.norm(g - o) / np.linalg.norm(o)))
    out["full_field_rel_l2_steps_1_2"] = live
    if F is not None:
        out["floor_rel_l2_steps_1_2"] = {f: [float(x) for x in F["floors"][:2, i]]
                                         for i, f in enumerate(FIELDS)}
        steps = int(F["steps"])
        sp = torch.from_numpy(F["sample_planes"]).cuda()
        sn = torch.from_numpy(F["sample_nodes"]).cuda()
        D.set_state(dn["u0"])
        verr = np.zeros(steps)
        perr = np.zeros(steps)
        pflo = np.zeros(steps)
        for s in range(steps):
            D.step(1)
            g = [D.field(i)[sp, sn].cpu().numpy() for i in range(4)]
            o = F["samples"][s]
            vs = max(np.max(np.abs(o[i])) for i in range(3))
            verr[s] = max(np.max(np.abs(g[i] - o[i])) for i in range(3)) / vs
            ps = np.max(np.abs(o[3]))
            perr[s] = np.max(np.abs(g[3] - o[3])) / ps
            pflo[s] = np.max(np.abs(F["vsamples"][s, 3] - o[3])) / ps
        run_floor = np.maximum.accumulate(pflo)
        out["sampled_steps"] = steps
        out["velocity_err_over_velocity_scale"] = {"step_1": float(verr[0]),
                                                   "step_10": float(verr[9]),
                                                   "step_100": float(verr[-1]),
                                                   "max": float(verr.max())}
        out["pressure_err"] = {"step_1": float(perr[0]), "step_100": float(perr[-1]),
                               "max": float(perr.max())}
        out["pressure_floor_running_max_step_100"] = float(run_floor[-1])
        out["pressure_err_over_10x_floor_max"] = float(np.max(perr / (10 * run_floor)))
    return out


def batch_leg(a, torch):
    """Uneven batch: 64 independent 2D problems (N_P 4..12, 4x4..20x20
    elements, aspect 1..4, lambda2 1e-2..1e2, half cylindrical), each solved
    once per run by one captured graph of fused launches (every kernel
    instance once per phase for all problems), the sweep choice per
    band-system class set by the library's autotuner (sx_batch_tune); FP64
    and mixed (one FP64 refinement pass), both against the oracle; the
    graph of per-problem launches on 4 lane streams timed beside it."""
    from oracle import oracle as O
    from semtex_amd.problems import uneven_batch
    from semtex_amd.solver import SX_FP64, SX_MIXED, Batch, Field, GpuMesh, ModalMatrixSys
    probs = uneven_batch()
    t0 = time.perf_counter()
    res = {}
    refs = []
    for p in probs:
        m = p["mesh"]
        refs.append(O.solve_modes(m, p["lambda2"], 0.0, p["forcing"][:, :m.nel * m.npnp])[0])

    def timed(B):
        B.run()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(a.batch_runs):
            B.run()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) / a.batch_runs

    for name, prec in (("fp64", SX_FP64), ("mixed", SX_MIXED)):
        items = []
        for p in probs:
            m = p["mesh"]
            gm = GpuMesh(m)
            M = ModalMatrixSys(p["lambda2"], 0.0, 0, 1, gm, precision=prec)
            u = Field(gm, 1)
            src = torch.zeros((1, m.plane_size), dtype=torch.float64, device="cuda")
            src[0, :m.nel * m.npnp] = torch.from_numpy(p["forcing"][0])
            items.append((M, u, src, gm))
        entries = [(M, u, src) for (M, u, src, _) in items]
        B = Batch(entries, refine_passes=2)
        ms_untuned = timed(B)
        tuned = B.tune(reps=5)
        ms = timed(B)
        err = max(float(np.linalg.norm(u.data[0, :p["mesh"].nel * p["mesh"].npnp].cpu().numpy()
                                       - r) / np.linalg.norm(r))
                  for (p, (_, u, _, _), r) in zip(probs, items, refs))
        res[name] = {"ms_per_run": round(ms, 4), "problems_per_s": round(len(probs) / (ms / 1e3), 1),
                     "ms_untuned": round(ms_untuned, 4), "max_rel_err_vs_oracle": err,
                     "plan": tuned}
        del B
        if name == "fp64":
            os.environ["SX_BATCH_FUSED"] = "0"
            B0 = Batch(entries, refine_passes=2)
            del os.environ["SX_BATCH_FUSED"]
            res["fp64_lane_graph_ms"] = round(timed(B0), 4)
            del B0
        del items, entries
    res["setup_s"] = round(time.perf_counter() - t0, 2)
    res["problems"] = len(probs)
    res["config"] = ("64 independent 2D Helmholtz problems, N_P 4..12, 4x4..20x20 elements, "
                     "aspect 1..4, lambda2 log-uniform 1e-2..1e2, N(0,1) forcing, half Cartesian "
                     "(Dirichlet), half cylindrical axisymmetric (axis y=0); one HIP graph per run "
                     "(fused launches, autotuned sweep choice); mixed: one FP64 refinement pass")
    return res


def adjoint_leg(torch, P, gm, reps=3):
    """Time of one gradient evaluation: (a) J = 1/2 ||u - u_t||_M^2 through
    the batched Helmholtz solve w.r.t. the forcing and lambda2; (b) the same
    J through 20 steps of the channel shrunk to 6x12 elements, N_P=6,
    N_Z=32, w.r.t. the initial field, checkpointed every 5 steps.  Median
    wall time of `reps` evaluations after one warm-up, synchronised."""
    from semtex_amd.adjoint import DnsTape
    from semtex_amd.problems import dns_channel
    from semtex_amd.solver import helmholtz_solve, mass_weight

    rng = np.random.default_rng(20261203)
    F = torch.from_numpy(P["forcing"]).cuda()
    Ut = torch.from_numpy(0.01 * rng.standard_normal(F.shape)).cuda()
    W = mass_weight(gm, torch.ones_like(F), 1.0)       # Q8 = Q4 (Cartesian)

    def grad_helmholtz():
        f = F.clone().requires_grad_(True)
        l2 = torch.tensor(P["lambda2"], dtype=torch.float64, requires_grad=True)
        u = helmholtz_solve(f, l2, gm, P["beta"], P["nmodes"])
        d = u - Ut
        J = 0.5 * (d * d * W).sum()
        J.backward()
        torch.cuda.synchronize()

    D = dns_channel(nx=6, ny=12, np_=6, nz=32)
    T = DnsTape(D["mesh_u"], D["mesh_p"], D["nz"], D["beta"], D["kinvis"], D["dt"],
                const_force=D["const_force"])
    Udt = torch.from_numpy(0.1 * rng.standard_normal((3, D["nz"], T.n))).cuda()

    def grad_dns():
        x = torch.from_numpy(D["u0"]).cuda().requires_grad_(True)
        st = T.run(x, 20, checkpoint=5)
        J = 0.5 * T.mass_norm2(st[0] - Udt)
        J.backward()
        torch.cuda.synchronize()

    def timed(fn):
        fn()
        ts = []
        for _ in range(reps):
            t0 = time.perf_counter()
            fn()
            ts.append(time.perf_counter() - t0)
        return round(1e3 * sorted(ts)[len(ts) // 2], 2)

    return {"helmholtz_grad_ms": timed(grad_helmholtz),
            "dns20_grad_ms": timed(grad_dns),
            "config": "(a) 16x16 N_P=10 N_Z=64 batch, d/df and d/dlambda2; (b) channel 6x12 "
                      "N_P=6 N_Z=32, 20 steps, d/du0, checkpoint every 5 steps"}


def main():
    a = parse()
    if a.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU only; --gpus must be 1"}))
        sys.exit(2)
    if a.cpu_dns_child:
        cpu_baseline_dns_child()
        return
    import torch

    if a.copy_calibration:
        copy_calibration(torch)
        return
    from semtex_amd import _lib
    from semtex_amd.problems import helmholtz_fourier
    from semtex_amd.solver import SX_FP64, SX_MIXED, GpuMesh

    assert torch.cuda.is_available(), "bench needs a GPU"
    L = _lib.load()
    P = helmholtz_fourier()
    m, nz, nmodes = P["mesh"], P["nz"], P["nmodes"]
    n = m.nel * m.npnp
    print(f"# mesh {m.info['nx']}x{m.info['ny']} np={m.np} nz={nz} nglobal={m.nglobal} "
          f"nsolve={m.nsolve} nband={m.nband} ({m.info['ordering']})", file=sys.stderr, flush=True)
    if a.dns_only:
        dn = dns_leg(a, torch)
        print(json.dumps({"dns_steps_per_s": round(dn["value"], 3),
                          "ms_per_step": round(dn["ms_per_step"], 4),
                          "steps": a.dns_steps, "finite": dn["finite"]}), flush=True)
        return
    gm = GpuMesh(m)
    f64 = helmholtz_leg(a, P, gm, SX_FP64, L, _lib, torch)
    print(f"# FP64: {f64['value']:.1f} mode-solves/s, {f64['ms_per_step']:.4f} ms/step, "
          f"setup {f64['setup_s']:.3f} s", file=sys.stderr, flush=True)
    planes = [k for k in range(nz) if k != 1]
    u64 = f64["solution"].cpu().numpy()[planes, :n]

    rel_err = None
    if not a.no_parity:
        from oracle import oracle as O
        om = O.OracleMesh(m)
        errs = []
        for md in (0, 1, nmodes - 1):
            S = O.OracleMsys(om, P["lambda2"], (P["beta"] * md) ** 2)
            for k in ([0] if md == 0 else [2 * md, 2 * md + 1]):
                uo = S.solve_plane(P["forcing"][k, :n])
                errs.append(np.linalg.norm(f64["solution"][k, :n].cpu().numpy() - uo)
                            / np.linalg.norm(uo))
        rel_err = float(max(errs))
        print(f"# parity vs oracle (modes 0,1,{nmodes-1}): max rel L2 {rel_err:.3e}",
              file=sys.stderr, flush=True)

    variants = {"fp64": {"value": round(f64["value"], 2),
                         "ms_per_step": round(f64["ms_per_step"], 5),
                         "rel_err_vs_oracle": rel_err}}
    value, chosen = f64["value"], "fp64"
    if not a.no_mixed:
        mx = helmholtz_leg(a, P, gm, SX_MIXED, L, _lib, torch)
        umx = mx["solution"].cpu().numpy()[planes, :n]
        err_mx = float(np.linalg.norm(umx - u64) / np.linalg.norm(u64))
        variants["mixed"] = {"value": round(mx["value"], 2),
                             "ms_per_step": round(mx["ms_per_step"], 5),
                             "refinement_iters": mx["iters"], "refine_tol": a.mixed_tol,
                             "rel_err_vs_fp64": err_mx,
                             "speedup_vs_fp64": round(mx["value"] / f64["value"], 3)}
        print(f"# mixed: {mx['value']:.1f} mode-solves/s, {mx['iters']} refinement passes, "
              f"rel err vs FP64 {err_mx:.2e}", file=sys.stderr, flush=True)
        if err_mx <= 1e-10 and mx["value"] > value:
            value, chosen = mx["value"], "mixed"
        del mx

    # bytes of one condensed solve: the dissection's operators of every mode
    # once (the band factor, 8 nsolve nband, where a system solves by it) and
    # its right-hand sides read and solutions written
    M = f64["M"]
    lay = M.layout()
    band_bytes = 0
    for md in range(nmodes):
        ns = M.nsolve(md)
        nrhs = 1 if md == 0 else 2
        factor = 8 * lay["operators"] if lay["kernel"] == 4 else 8 * ns * m.nband
        band_bytes += factor + 16 * ns * nrhs
    phases = f64["phases"]
    band_ms = phases["band_solve"]
    achieved = band_bytes / (band_ms * 1e-3) / 1e9

    workload = ("batched 2.5D Helmholtz, 16x16 elements on [0,2pi]x[-1,1], N_P=10, "
                "N_Z=64 (32 modes, beta=1, lambda2=1+k^2), Dirichlet y=+-1, periodic x, "
                "seeded Gaussian forcing ~(1+k)^-2; static condensation + direct solve by dissection")
    out = {
        "metric": METRIC,
        "value": round(value, 2),
        "unit": "mode-solves/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": round(nmodes / value * 1e3, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {
            "workload": workload,
            "precision": chosen,
            "mode_solves_per_step": nmodes,
            "nglobal": m.nglobal, "nsolve": m.nsolve, "nband": m.nband,
            "ordering": m.info["ordering"],
        },
        "variants": variants,
        "roofline": {
            "kernel": "k_tree_level" if lay["kernel"] == 4 else "k_band_solve",
            "bound": "hbm",
            "achieved": round(achieved, 1),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4),
            "traffic": None,
            "algorithmic_bytes": band_bytes,
            "avg_ms": round(band_ms, 5),
        },
        "phases_ms": {k: round(v, 5) for k, v in phases.items()},
        "setup_s": round(f64["setup_s"], 3),
        "rel_err_vs_oracle": rel_err,
        "wall_s_timed": round(f64["wall_s"], 4),
    }
    del f64

    if not a.no_dns:
        dn = dns_leg(a, torch)
        dns = {"value": round(dn["value"], 3), "unit": "DNS steps/s",
               "ms_per_step": round(dn["ms_per_step"], 4), "steps": a.dns_steps,
               "warmup": a.dns_warmup, "setup_s": round(dn["setup_s"], 3),
               "finite": dn["finite"],
               "config": "forced channel 12x24 elements on [0,4pi]x[-1,1], N_P=8, N_Z=128, "
                         "Lz=2pi, Re=2000, dt=1e-3, SS2 splitting, skew-symmetric advection, "
                         "Poiseuille + U(-1e-2,1e-2) perturbation (seeded), FP64"}
        dns["roofline"] = dns_roofline(dn)
        if not a.no_cpu_baseline:
            cb = cpu_baseline_dns()
            cb["value"] = round(cb["value"], 4)
            dns["cpu_baseline"] = cb
            dns["gpu_over_cpu"] = round(dn["value"] / cb["value"], 1)
        if not a.no_parity:
            dns["parity"] = dns_parity(dn, torch)
        if not a.no_dealias:
            dl = dns_leg(a, torch, dealias=True)
            dns["dealiased"] = {"value": round(dl["value"], 3),
                                "ms_per_step": round(dl["ms_per_step"], 4),
                                "finite": dl["finite"],
                                "config": "same channel, 3/2-rule dealiased products (M = 192 "
                                          "z planes), skew-symmetric advection"}
            del dl
        out["dns"] = dns
        print(f"# DNS: {dn['value']:.2f} steps/s ({dn['ms_per_step']:.3f} ms/step)",
              file=sys.stderr, flush=True)

    if not a.no_batch:
        out["batch"] = batch_leg(a, torch)
        print(f"# batch: {out['batch']['fp64']['problems_per_s']} problems/s FP64, "
              f"{out['batch']['mixed']['problems_per_s']} mixed; lane graph "
              f"{out['batch']['fp64_lane_graph_ms']} ms", file=sys.stderr, flush=True)

    if not a.no_adjoint:
        out["adjoint"] = adjoint_leg(torch, P, gm)
        print(f"# adjoint: {out['adjoint']}", file=sys.stderr, flush=True)

    if not a.no_cpu_baseline:
        cb = cpu_baseline(P, a.cpu_seconds)
        cb["value"] = round(cb["value"], 2)
        out["cpu_baseline"] = cb
        out["gpu_over_cpu"] = round(value / cb["value"], 1)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
