"""Benchmark of the DMRG two-site H*psi hot path on one MI355X.

Workload (one "step"): one dense two-site effective-Hamiltonian product
H*psi = noPrime(((psi*L)*W1)*W2*R) with psi in R^{chi x 2 x 2 x chi},
L, R in R^{chi x 5 x chi}, W1 = W2 = the bulk Heisenberg MPO tensor
(5 x 2 x 2 x 5), chi = 1024, entries of psi, L, R i.i.d. N(0,1) from a fixed
seed (synthetic data), all operands resident in HBM before timing.
The contractions run through the libitx C ABI (plans built once), in the
order LocalOp::product runs them: psi*L, then the MPO pair pre-contracted
(W12 = W1*W2, same flop count and result layout), then *R (--chain 4stage
runs the reference's four separate stages instead).

value = algorithmic FP64-equivalent flops (80 chi^3 + 800 chi^2 per H*psi)
        / wall time, whole job (one GPU).

Further legs on the same line: "qn_hpsi" -- the block-sparse H*psi at
chi = 1024 over 31 Sz sectors in every execution mode (grouped chain as a
HIP graph / launched directly / eager, one launch per block pair, FP32 and
BF16x3 forms); "dmrg" -- QN Heisenberg DMRG N=100 with the maxdim ramp to
2048 (cutoff 1e-10) in the FP64, FP32 and BF16x3 H*psi forms: seconds per
sweep, energies and their differences; "dmrg_big" -- the same chain with
MinDim = MaxDim along a ramp to 1024; "hubbard" -- the 8 x 4 Hubbard
cylinder at maxdim 400; "hubbard_big" -- the cylinder along the maxdim ramp
to 2500.

usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--chi 1024]
                       [--no-cpu] [--no-qn] [--dmrg N:maxdims|''] [--dmrg-forms f64,f32,bf16x3]
                       [--prec f64|f32|bf16x3] [--chain fused|4stage]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "DMRG sec/sweep + Hψ TFLOP/s, mixed vs FP64 on 1 MI355X at |ΔE|≤1e-9"
# TFLOP/s dense MFMA (datasheet); the BF16x3 form runs 3 BF16 products per
# FP64-equivalent product, so its FP64-equivalent ceiling is 2500/3
PEAK = {"f64": 78.6, "f32": 157.3, "bf16x3": 2500.0 / 3, "bf16x3s": 2500.0 / 3}
SEED = 20261202 + 2

from itensor_amd.workloads import (DMRG_BIG_MAXDIM, DMRG_MAXDIM, FUSED, HUBBARD_BIG_MAXDIM, HUBBARD_MAXDIM,  # noqa: E402
                                   SECTORS_1024, STAGES,
                                   fused_dims, heisenberg_qn_chain, heisenberg_w, hpsi_flops, hubbard_cylinder,
                                   qn_operands, stage_dims)


def cpu_baseline(psi, L, W, R, budget_s: float = 20.0):
    """The oracle's H*psi (numpy tensordot over the host BLAS) on the host
    cores: 1 warm-up, then repeats until ~budget_s, median reported."""
    from oracle.dense import hpsi_dense

    threads, _, _ = host_cpu()
    t0 = time.perf_counter()
    ref = hpsi_dense(psi, L, W, W, R)
    first = time.perf_counter() - t0
    times = []
    reps = max(1, min(5, int(budget_s / max(first, 1e-3))))
    for _ in range(reps):
        t0 = time.perf_counter()
        hpsi_dense(psi, L, W, W, R)
        times.append(time.perf_counter() - t0)
    return ref, float(np.median(times)), threads, reps


def qn_hpsi(steps: int, warmup: int):
    """Block-sparse H*psi (chi = 1024 over 31 Sz sectors) through
    LocalOp::product in each execution mode: the grouped-GEMM chain
    replayed as a HIP graph, the same chain launched directly, eager
    operator* products, and one launch per block pair (the reference's
    loop).  Wall time per product over `steps` products after `warmup`."""
    import torch

    from itensor_amd import host as H

    phi, L, W1, W2, R = qn_operands(H, SECTORS_1024, 20261202 + 3)
    modes = [("graph", H.HPSI_GRAPH, 0), ("planned", H.HPSI_PLANNED, 0), ("eager", H.HPSI_EAGER, 0),
             ("per_block", H.HPSI_PER_BLOCK, 0), ("graph_f32", H.HPSI_GRAPH, 1),
             ("graph_bf16x3", H.HPSI_GRAPH, 2)]
    res, ref = {}, None
    for name, mode, prec in modes:
        op = H.LocalOp(W1, W2, L, R, True)
        op.set_mode(mode)
        op.set_precision(prec)
        flops = op.flops(phi) if mode != H.HPSI_EAGER else res["graph"]["flops"]
        t_plan = time.perf_counter()
        out = op.product(phi)
        torch.cuda.synchronize()
        t_plan = time.perf_counter() - t_plan
        for _ in range(warmup):
            op.product(phi)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            op.product(phi)
        torch.cuda.synchronize()
        ms = (time.perf_counter() - t0) / steps * 1e3
        st = out.store()
        tf = flops / (ms * 1e-3) / 1e12
        form = ("f64", "f32", "bf16x3")[prec]
        r = {"ms_per_hpsi": round(ms, 4), "tflops": round(tf, 3), "flops": flops,
             "frac_of_peak": round(tf / PEAK[form], 4), "first_call_ms": round(t_plan * 1e3, 2)}
        if ref is None:
            ref = (st, out.offsets)
            r["blocks_out"] = len(out.offsets)
        else:
            r["same_block_list"] = out.offsets == ref[1]
            r["rel_err_vs_graph_f64"] = float(np.max(np.abs(st - ref[0])) / np.max(np.abs(ref[0])))
        res[name] = r
    res["blocks_phi"] = len(phi.offsets)
    res["speedup_grouped_vs_per_block"] = round(res["per_block"]["ms_per_hpsi"] / res["graph"]["ms_per_hpsi"], 2)
    return res




def _leg_summary(E, recs, secs, wall, nsweeps):
    last = [r for r in recs if r["sweep"] == nsweeps]
    fl = np.sum([r["hpsi_flops"] for r in recs], axis=0)
    return {"energy": E, "wall_s": round(wall, 3), "sec_per_sweep": [round(x, 4) for x in secs],
            "max_dim": [max(r["dim"] for r in recs if r["sweep"] == k + 1) for k in range(nsweeps)],
            "truncerr_max_last_sweep": max(r["truncerr"] for r in last),
            "hpsi_products_last_sweep": sum(r["nprod"] for r in last),
            # share of the H*psi flops whose kernels computed in each form
            "hpsi_flops_by_form": {k: round(float(v / max(fl.sum(), 1.0)), 4)
                                   for k, v in zip(("f64", "f32", "bf16x3"), fl)},
            "hpsi_flops_total": float(fl.sum())}


def _phase_split(recs, nsweeps):
    last = [r for r in recs if r["sweep"] == nsweeps]
    return {"env": round(sum(r["t_env"] for r in last), 4), "davidson": round(sum(r["t_davidson"] for r in last), 4),
            "svd": round(sum(r["t_svd"] for r in last), 4)}


def dmrg_leg(N: int, maxdims, prec: int, mode: int, final_fp64: int = 0, mindim_follows: bool = False,
             sync_timing: bool = False):
    """QN Heisenberg DMRG (N sites, Neel start, one sweep per maxdim entry,
    cutoff 1e-10, Davidson niter 2) in one H*psi form: wall time of each
    sweep (everything included, no added synchronisation).  With
    mindim_follows, MinDim = MaxDim so that the bond dimension follows the
    ramp instead of saturating at the cutoff.  With sync_timing, the device
    is synchronised between the phases of every bond step and the phase
    split of the last sweep is reported (a diagnostic run, slower)."""
    import torch

    from itensor_amd import host as H

    mpo, A = heisenberg_qn_chain(H, N)
    sweeps = [{"MaxDim": int(m), "MinDim": int(m) if mindim_follows else 1, "Cutoff": 1e-10, "Niter": 2}
              for m in maxdims]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    E, recs, _, secs = H.dmrg(mpo, A, sweeps, {"HpsiPrecision": prec, "HpsiMode": mode, "SyncTiming": sync_timing,
                                               "FinalFP64Sweeps": final_fp64})
    wall = time.perf_counter() - t0
    out = _leg_summary(E, recs, secs, wall, len(maxdims))
    if sync_timing:
        out["last_sweep_split_s"] = _phase_split(recs, len(maxdims))
    return out


def hubbard_leg(Nx: int, Ny: int, maxdims, prec: int, final_fp64: int = 0, sync_timing: bool = False):
    """(Nf, Sz)-conserving Hubbard DMRG on the Nx x Ny YPeriodic cylinder
    (t = 1, U = 4, half filling, cutoff 1e-9, niter 2, noise 1e-6 / 1e-7 on
    the first two sweeps) in one H*psi form: wall time per sweep."""
    import torch

    from itensor_amd import host as H

    mpo, A = hubbard_cylinder(H, Nx, Ny, 1.0, 4.0, True)
    noise = [1e-6, 1e-7] + [0.0] * max(0, len(maxdims) - 2)
    sweeps = [{"MaxDim": int(m), "Cutoff": 1e-9, "Niter": 2, "Noise": z} for m, z in zip(maxdims, noise)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    E, recs, _, secs = H.dmrg(mpo, A, sweeps, {"HpsiPrecision": prec, "SyncTiming": sync_timing,
                                               "FinalFP64Sweeps": final_fp64})
    wall = time.perf_counter() - t0
    out = _leg_summary(E, recs, secs, wall, len(maxdims))
    if sync_timing:
        out["last_sweep_split_s"] = _phase_split(recs, len(maxdims))
    return out


def host_cpu():
    """(BLAS threads the host oracle runs with, cores this process may use,
    CPU model).  The BLAS thread count is what the numpy legs use; the
    oracle's Python loops around it run on one core."""
    try:
        nproc = len(os.sched_getaffinity(0))
    except AttributeError:  # pragma: no cover
        nproc = os.cpu_count() or 1
    try:
        from threadpoolctl import threadpool_info

        threads = max([i.get("num_threads", 1) for i in threadpool_info()] or [1])
    except Exception:  # pragma: no cover
        threads = nproc
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return threads, nproc, model


def cpu_qn_hpsi(budget_s: float = 10.0):
    """The oracle's block-sparse H*psi (per-block numpy loop, the
    reference's doTask loop restated) on the chi = 1024 / 31-sector operands
    on the host cores: median of repeats within budget_s."""
    from oracle.dmrg import local_op_product
    from tests.hpsi_cases import hpsi_operands

    phi, L, W1, W2, R = hpsi_operands(SECTORS_1024, seed=20261202 + 3)
    t0 = time.perf_counter()
    local_op_product(phi, L, W1, W2, R)
    first = time.perf_counter() - t0
    times = []
    for _ in range(max(1, min(20, int(budget_s / max(first, 1e-3))))):
        t0 = time.perf_counter()
        local_op_product(phi, L, W1, W2, R)
        times.append(time.perf_counter() - t0)
    return float(np.median(times)), len(times)


def cpu_dmrg(N: int, maxdims):
    """The oracle's QN DMRG (numpy restatement of DMRGWorker, davidson and
    denmatDecomp) on the host cores for the first sweeps of the ramp: wall
    time per sweep."""
    from oracle import dmrg as OD

    sites = OD.spin_half_sites(N, True)
    Hm = OD.heisenberg_mpo(sites)
    psi = OD.product_mps(sites, [i % 2 for i in range(N)])
    secs, E = [], None
    for m in maxdims:
        t0 = time.perf_counter()
        E, psi = OD.dmrg(Hm, psi, [{"MaxDim": m, "Cutoff": 1e-10, "Niter": 2}])
        secs.append(time.perf_counter() - t0)
    return secs, E


# kernels of the engine's tile indices that differ from the generic MFMA tile
KERNEL_OF_TILE = {5: "k_skinny", 10: "k_small", 14: "k_pipe", 15: "k_pipe", 16: "k_pipe", 17: "k_pipe", 18: "k_pipe"}


def measured_traffic(chi: int, prec: str, stage: str):
    """HBM bytes per launch of a stage as rocprofv3 FETCH_SIZE + WRITE_SIZE
    measured them (copy-calibrated) -- read from the committed profile
    summary of the chi = 1024 FP64 chain; None for other workloads."""
    if chi != 1024 or prec != "f64":
        return None
    path = os.path.join(ROOT, "profiles", "pmc_dense_hpsi_chi1024.md")
    try:
        import re

        m = re.search(r"traffic_bytes_per_launch %s = (\d+)" % stage, open(path).read())
        return int(m.group(1)) if m else None
    except OSError:
        return None


def copy_calibration(gib: float):
    """A plain device-to-device copy of known size (reads and writes
    `gib` GiB per launch), the reference point for HBM byte counters."""
    import torch

    import itensor_amd  # noqa: F401

    n = int(gib * (1 << 30) / 8)
    x = torch.ones(n, dtype=torch.float64, device="cuda:0")
    y = torch.empty_like(x)
    for _ in range(5):
        y.copy_(x)
    torch.cuda.synchronize()
    print(json.dumps({"calibration": "device copy", "bytes_read": n * 8, "bytes_written": n * 8, "launches": 5}))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--chi", type=int, default=1024)
    ap.add_argument("--prec", default="f64", choices=["f64", "f32", "bf16x3"])
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--chain", default="fused", choices=["fused", "4stage"],
                    help="LocalOp::product as run by the host layer (MPO pair fused) or the 4-stage chain")
    ap.add_argument("--no-qn", action="store_true", help="skip the block-sparse (31 Sz sectors) H*psi leg")
    ap.add_argument("--dmrg", default="100:full",
                    help="QN DMRG leg: N:maxdim1,maxdim2,... ('full' = the 10-sweep ramp to 2048); '' skips it")
    ap.add_argument("--dmrg-forms", default="f64,f32,bf16x3,bf16x3+f64last",
                    help="H*psi forms of the DMRG leg ('+f64last': the last sweep in FP64)")
    ap.add_argument("--hubbard", default="8x4:" + ",".join(str(m) for m in HUBBARD_MAXDIM),
                    help="Hubbard cylinder leg: NxxNy:maxdim1,maxdim2,... ('' skips it)")
    ap.add_argument("--hubbard-forms", default="f64,f32,bf16x3+f64last",
                    help="H*psi forms of the Hubbard leg ('+f64last': the last sweep in FP64)")
    ap.add_argument("--hubbard-big", default="8x4:" + ",".join(str(m) for m in HUBBARD_BIG_MAXDIM),
                    help="Hubbard cylinder leg along the maxdim ramp toward 4096 ('' skips it)")
    ap.add_argument("--hubbard-big-forms", default="f64,f32", help="H*psi forms of that leg")
    ap.add_argument("--dmrg-big", default="100:" + ",".join(str(m) for m in DMRG_BIG_MAXDIM),
                    help="QN DMRG leg with MinDim = MaxDim (the bond dimension follows the ramp; 'full' = the ramp "
                         "to 2048); '' skips it")
    ap.add_argument("--dmrg-big-forms", default="f64,f32,bf16x3",
                    help="H*psi forms of the MinDim = MaxDim DMRG leg")
    ap.add_argument("--phase-split", action="store_true",
                    help="also run each DMRG workload once in FP64 with a synchronised phase split")
    ap.add_argument("--copy-gib", type=float, default=0.0,
                    help="calibration only: time a plain device copy of this many GiB (for PMC byte counters)")
    args = ap.parse_args()
    if args.copy_gib > 0:
        return copy_calibration(args.copy_gib)
    if args.gpus != 1:
        print(json.dumps({"error": "this build measures one GPU only; --gpus must be 1",
                          "n_gpus_requested": args.gpus}))
        sys.exit(2)

    import torch

    from itensor_amd.itx import Context

    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU visible"}))
        sys.exit(1)
    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream()
    ctx = Context(0, stream.cuda_stream)
    ctx.set_autotune(True)  # tile shapes measured per size class at plan creation (untimed)

    chi = args.chi
    rng = np.random.default_rng(SEED)
    psi = rng.standard_normal((chi, 2, 2, chi))
    L = rng.standard_normal((chi, 5, chi))
    R = rng.standard_normal((chi, 5, chi))
    W = heisenberg_w()

    def put(a):
        return torch.from_numpy(np.ascontiguousarray(a.ravel(order="F"))).to(dev)

    d_psi, d_L, d_R, d_W = put(psi), put(L), put(R), put(W)
    if args.chain == "fused":
        W12 = np.einsum("aijb,bklc->aijklc", W, W)  # W1*W2 over h1: (h0,s1,s1',s2,s2',h2)
        dims, labels = fused_dims(chi), FUSED
        ops = [d_L, put(W12), d_R]
    else:
        dims, labels = stage_dims(chi), STAGES
        ops = [d_L, d_W, d_W, d_R]
    nst = len(dims)
    bufs = [torch.empty(int(np.prod(dc)), dtype=torch.float64, device=dev) for (_, _, dc) in dims]
    inputs = [d_psi] + bufs[:-1]

    def run_forms(prec):
        if prec == "bf16x3s":  # BF16x3 with pre-split operands on the MFMA stages
            plans = [ctx.plan_dense(da, la, db, lb, dc, lc, "bf16x3" if i != 1 else "f64")
                     for i, ((da, db, dc), (la, lb, lc)) in enumerate(zip(dims, labels))]
            for i in (0, len(plans) - 1):
                plans[i].set_split(True)
            return plans
        return [ctx.plan_dense(da, la, db, lb, dc, lc, prec) for (da, db, dc), (la, lb, lc) in zip(dims, labels)]

    # Pre-split form (fused chain): L and R are split once, as the
    # environments of a Davidson call are; psi and the MPO stage's output are
    # split inside every step (their passes timed as their own stages).
    split_form = args.chain == "fused"
    if split_form:
        def words(n):
            return torch.empty(n, dtype=torch.int32, device=dev)

        w_in = [words(d_psi.numel()), None, words(bufs[1].numel())]
        w_op = [words(d_L.numel()), None, words(d_R.numel())]
        ctx.split_bf16(d_L.data_ptr(), w_op[0].data_ptr(), d_L.numel())
        ctx.split_bf16(d_R.data_ptr(), w_op[2].data_ptr(), d_R.numel())

    def launches(prec, plans):
        """The step as a list of launches (name, callable)."""
        if prec != "bf16x3s":
            return [("S%d" % (i + 1), (lambda p=p, a=a, b=b, c=c: p.execute(a.data_ptr(), b.data_ptr(), c.data_ptr())))
                    for i, (p, a, b, c) in enumerate(zip(plans, inputs, ops, bufs))]
        out = []
        for i, (p, a, b, c) in enumerate(zip(plans, inputs, ops, bufs)):
            if i == 1:
                out.append(("S2", lambda p=p, a=a, b=b, c=c: p.execute(a.data_ptr(), b.data_ptr(), c.data_ptr())))
                continue
            out.append(("split%d" % (i + 1), lambda a=a, w=w_in[i]: ctx.split_bf16(a.data_ptr(), w.data_ptr(), a.numel())))
            out.append(("S%d" % (i + 1),
                        lambda p=p, wa=w_in[i], wb=w_op[i], c=c: p.execute(wa.data_ptr(), wb.data_ptr(), c.data_ptr())))
        return out

    results = {}
    flops = hpsi_flops(chi)
    forms_run = [args.prec] + [p for p in ("f64", "f32", "bf16x3") if p != args.prec]
    if split_form:
        forms_run.append("bf16x3s")
    for prec in forms_run:
        plans = run_forms(prec)
        steps = launches(prec, plans)
        for _ in range(args.warmup):
            for _, f in steps:
                f()
        torch.cuda.synchronize()
        # whole-step timing (wall clock around K steps)
        t0 = time.perf_counter()
        for _ in range(args.steps):
            for _, f in steps:
                f()
        torch.cuda.synchronize()
        wall = time.perf_counter() - t0
        # per-launch HIP-event timing on the stream the kernels run on
        nl = len(steps)
        ev = [[torch.cuda.Event(enable_timing=True) for _ in range(nl + 1)] for _ in range(args.steps)]
        for s in range(args.steps):
            for i, (_, f) in enumerate(steps):
                ev[s][i].record(stream)
                f()
            ev[s][nl].record(stream)
        torch.cuda.synchronize()
        launch_ms = {name: float(np.mean([ev[s][i].elapsed_time(ev[s][i + 1]) for s in range(args.steps)]))
                     for i, (name, _) in enumerate(steps)}
        stage_ms = [launch_ms["S%d" % (i + 1)] for i in range(nst)]
        out = bufs[-1].detach().cpu().numpy().reshape((chi, 2, 2, chi), order="F")
        results[prec] = {"wall_s": wall, "stage_ms": stage_ms, "out": out,
                         "stage_flops": [p.flops for p in plans],
                         "stage_tiles": [p.info["tile"] for p in plans],
                         "split_ms": {k: v for k, v in launch_ms.items() if k.startswith("split")}}
        for p in plans:
            p.close()

    main_r = results[args.prec]
    ms = main_r["wall_s"] / args.steps * 1e3
    value = flops / (ms * 1e-3) / 1e12

    # dominant kernel: the stage with the largest average duration
    st = main_r["stage_ms"]
    dom = int(np.argmax(st))
    dom_flops = main_r["stage_flops"][dom]
    achieved = dom_flops / (st[dom] * 1e-3) / 1e12

    line = {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": args.prec,
        "data": "synthetic (psi, L, R iid N(0,1), seed %d; Heisenberg W)" % SEED,
        "config": {"workload": "dense two-site Hpsi, chi=%d, d=2, k=5 (Heisenberg MPO)" % chi,
                   "chi": chi, "flops_per_step": flops, "chain": args.chain, "parallelism": "single GPU"},
        "roofline": {"bound": "mfma", "achieved": round(achieved, 3), "peak": PEAK[args.prec],
                     "unit": "TFLOP/s", "frac": round(achieved / PEAK[args.prec], 4),
                     "traffic": measured_traffic(chi, args.prec, ["S1", "W12", "S4"][dom] if nst == 3 else "none"),
                     "traffic_source": "profiles/pmc_dense_hpsi_chi1024.md (rocprofv3 FETCH_SIZE + WRITE_SIZE per "
                                       "dispatch, scaled by a 1 GiB copy: x2.0 / x1.0)",
                     "kernel": "%s (stage %d of %d of H*psi, tile %d)" % (
                         "k_dgemm" if args.prec == "f32" and main_r["stage_tiles"][dom] in (14, 15) else
                         KERNEL_OF_TILE.get(main_r["stage_tiles"][dom], "k_gemm"), dom + 1, nst,
                         main_r["stage_tiles"][dom]),
                     "flops_per_launch": dom_flops, "avg_launch_ms": round(st[dom], 4)},
        "stages_ms": {args.prec: [round(x, 4) for x in st]},
        "forms": {},
        # where this build's path differs from the north star's letter or the reference's algorithm
        "deviations": [
            "Davidson's small Rayleigh-Ritz eigenproblem (at most (niter+2)^2) is solved on the host in FP64",
            "the density-matrix eigensolver runs on the device by divide and conquer up to 512 rows; "
            "larger blocks go to rocSOLVER dsyevd",
            "the Hubbard MPO is the host AutoMPO's exact finite-state-machine MPO, not the reference's "
            "SVD-compressed one: the same operator, other link sectors",
            "a reduced-precision sweep reports the FP64 Rayleigh quotient of its last Ritz vector",
        ],
    }
    for prec, r in results.items():
        line["stages_ms"][prec] = [round(x, 4) for x in r["stage_ms"]]
        sm = r["stage_ms"]
        dk = int(np.argmax(sm))
        ach = r["stage_flops"][dk] / (sm[dk] * 1e-3) / 1e12
        line["forms"][prec] = {"tflops": round(flops / (r["wall_s"] / args.steps) / 1e12, 3),
                               "ms_per_hpsi": round(r["wall_s"] / args.steps * 1e3, 4),
                               # the form's dominant stage against the peak of the arithmetic it runs on
                               # (BF16x3: three BF16 products per FP64-equivalent one)
                               "roofline": {"bound": "mfma", "achieved": round(ach, 3), "peak": PEAK[prec],
                                            "unit": "TFLOP/s (FP64-equivalent)", "frac": round(ach / PEAK[prec], 4),
                                            "stage": dk + 1, "avg_launch_ms": round(sm[dk], 4)}}
        if r["split_ms"]:
            line["forms"][prec]["split_pass_ms"] = {k: round(v, 4) for k, v in r["split_ms"].items()}
            if "bf16x3" in results:
                line["forms"][prec]["bitwise_equal_to_bf16x3"] = bool(np.array_equal(r["out"], results["bf16x3"]["out"]))

    cores, nproc, cpu_model = host_cpu()
    cpu_model = "%s (%d cores visible)" % (cpu_model, nproc)
    if not args.no_qn:
        q = qn_hpsi(max(5, args.steps), args.warmup)
        line["qn_hpsi"] = {"workload": "block-sparse two-site Hpsi, chi=1024 over 31 Sz sectors "
                                       "(max 120, min 1), site {+1,-1}, MPO link {0:3,-2:1,+2:1}", **q}
        if not args.no_cpu:
            t_q, reps = cpu_qn_hpsi()
            qf = q["graph"]["flops"]
            line["qn_hpsi"]["cpu_baseline"] = {
                "value": round(qf / t_q / 1e12, 6), "unit": "TFLOP/s", "cores": cores, "kind": "port",
                "cpu": cpu_model,
                "sample": "oracle local_op_product (per-block numpy loop) on the same structure, median of %d: "
                          "%.4f s per H*psi" % (reps, t_q)}

    def mixed_deltas(res, forms):
        if "f64" in res:
            for form in forms:
                if form != "f64" and form in res:
                    res["dE_%s_vs_f64" % form] = res[form]["energy"] - res["f64"]["energy"]
                    res["sweep_speedup_%s_vs_f64" % form] = round(res["f64"]["wall_s"] / res[form]["wall_s"], 3)

    if args.dmrg:
        n_s, md_s = args.dmrg.split(":")
        mds = DMRG_MAXDIM if md_s == "full" else [int(x) for x in md_s.split(",")]
        forms = args.dmrg_forms.split(",")
        dm = {"workload": "QN Heisenberg N=%s open chain (total Sz 0, Neel start), maxdim %s, cutoff 1e-10, "
                          "niter 2; H*psi in the named form, everything else FP64; sec/sweep without added "
                          "synchronisation" % (n_s, mds)}
        for form in forms:
            base, _, last = form.partition("+")
            dm[form] = dmrg_leg(int(n_s), mds, {"f64": 0, "f32": 1, "bf16x3": 2}[base], 2,
                                1 if last == "f64last" else 0)
            print("dmrg leg %s done in %.1f s" % (form, dm[form]["wall_s"]), file=sys.stderr, flush=True)
        mixed_deltas(dm, forms)
        dm["phase_split_f64"] = dmrg_leg(int(n_s), mds, 0, 2, sync_timing=True)["last_sweep_split_s"]
        if not args.no_cpu:
            k = 3
            secs, e_cpu = cpu_dmrg(int(n_s), mds[:k])
            dm["cpu_baseline"] = {
                "value": round(secs[-1], 3), "unit": "s/sweep (maxdim %d)" % mds[k - 1], "cores": cores,
                "kind": "port", "cpu": cpu_model,
                "sample": "oracle dmrg (numpy restatement of DMRGWorker, davidson, denmatDecomp) on the same "
                          "chain, sweeps 1-%d of the ramp (maxdim %s): %s s per sweep; the GPU FP64 run's same "
                          "sweeps: %s s" % (k, mds[:k], [round(x, 3) for x in secs],
                                            dm.get("f64", {}).get("sec_per_sweep", [])[:k])}
        line["dmrg"] = dm
    if args.dmrg_big:
        n_s, md_s = args.dmrg_big.split(":")
        mds = DMRG_MAXDIM if md_s == "full" else [int(x) for x in md_s.split(",")]
        forms = args.dmrg_big_forms.split(",")
        db = {"workload": "QN Heisenberg N=%s open chain, MinDim = MaxDim = %s (the bond dimension follows the "
                          "ramp to its maximum instead of saturating at the cutoff), cutoff 1e-10, niter 2, "
                          "density-matrix bond step; H*psi in the named form" % (n_s, mds)}
        for form in forms:
            base, _, last = form.partition("+")
            db[form] = dmrg_leg(int(n_s), mds, {"f64": 0, "f32": 1, "bf16x3": 2}[base], 2,
                                1 if last == "f64last" else 0, mindim_follows=True)
            print("dmrg_big leg %s done in %.1f s" % (form, db[form]["wall_s"]), file=sys.stderr, flush=True)
        mixed_deltas(db, forms)
        if args.phase_split:
            db["phase_split_f64"] = dmrg_leg(int(n_s), mds, 0, 2, mindim_follows=True,
                                             sync_timing=True)["last_sweep_split_s"]
        line["dmrg_big"] = db

    if args.hubbard:
        geo, md_s = args.hubbard.split(":")
        nx, ny = (int(x) for x in geo.split("x"))
        mds = [int(x) for x in md_s.split(",")]
        forms = args.hubbard_forms.split(",")
        hb = {"workload": "Hubbard %dx%d YPeriodic cylinder (squareLattice order), t=1, U=4, half filling, "
                          "(Nf, Sz) QNs, MPO from the host AutoMPO; maxdim %s, cutoff 1e-9, niter 2, noise 1e-6/1e-7 "
                          "on the first two sweeps; H*psi in the named form, everything else FP64" % (nx, ny, mds)}
        for form in forms:
            base, _, last = form.partition("+")
            hb[form] = hubbard_leg(nx, ny, mds, {"f64": 0, "f32": 1, "bf16x3": 2}[base], 1 if last == "f64last" else 0)
            print("hubbard leg %s done in %.1f s" % (form, hb[form]["wall_s"]), file=sys.stderr, flush=True)
        mixed_deltas(hb, forms)
        if args.phase_split:
            hb["phase_split_f64"] = hubbard_leg(nx, ny, mds, 0, sync_timing=True)["last_sweep_split_s"]
        line["hubbard"] = hb

    if args.hubbard_big:
        geo, md_s = args.hubbard_big.split(":")
        nx, ny = (int(x) for x in geo.split("x"))
        mds = [int(x) for x in md_s.split(",")]
        forms = args.hubbard_big_forms.split(",")
        hg = {"workload": "Hubbard %dx%d YPeriodic cylinder, t=1, U=4, half filling, (Nf, Sz) QNs, maxdim ramp %s "
                          "(toward 4096; stopped at %d to fit the benchmark's time budget), cutoff 1e-9, niter 2, "
                          "noise 1e-6/1e-7 on the first two sweeps" % (nx, ny, mds, mds[-1])}
        for form in forms:
            base, _, last = form.partition("+")
            hg[form] = hubbard_leg(nx, ny, mds, {"f64": 0, "f32": 1, "bf16x3": 2}[base], 1 if last == "f64last" else 0)
            print("hubbard_big leg %s done in %.1f s" % (form, hg[form]["wall_s"]), file=sys.stderr, flush=True)
        mixed_deltas(hg, forms)
        line["hubbard_big"] = hg

    if not args.no_cpu:
        ref, t_cpu, threads, reps = cpu_baseline(psi, L, W, R)
        line["cpu_baseline"] = {"value": round(flops / t_cpu / 1e12, 5), "unit": "TFLOP/s",
                                "cores": threads, "kind": "port", "cpu": cpu_model,
                                "sample": "oracle hpsi_dense (numpy tensordot over the host BLAS) on the same "
                                          "chi=%d inputs, median of %d after 1 warm-up, %.3f s per H*psi"
                                          % (chi, reps, t_cpu)}
        nref = np.max(np.abs(ref))
        for prec, r in results.items():
            line["forms"][prec]["rel_err_vs_fp64_cpu"] = float(np.max(np.abs(r["out"] - ref)) / nref)
            line["forms"][prec]["rel_l2_err_vs_fp64_cpu"] = float(np.linalg.norm(r["out"] - ref) / np.linalg.norm(ref))
    print(json.dumps(line), flush=True)
    ctx.close()


if __name__ == "__main__":
    main()
