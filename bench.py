#!/usr/bin/env python3
"""Headline benchmark: one SpAMM multiply per step on one MI355X.

Workload (BASELINE.json metric: "SpAMM ms + effective TFLOP/s (kept tiles) at
N=16384 fp16, fixed tau"): N = 16384, tile 64, A and B independent seeded
exponential-decay matrices u_ij * exp(-lam |i-j|), fp32 in HBM, tau fixed
before the timed region so that ~10 % of the tile products are kept.
exp(-0.1 d) as literally written keeps < 0.1 % after fp16 rounding whatever
tau > 0 is chosen, so the timed workload uses lam = 0.003 (10 % reachable) and
the literal rate is run once and reported under "literal_config".

A step = spamm_multiply = convert+norm-map(B), convert+norm-map(A), gate,
gated GEMM, inputs already resident in HBM.  value = kept products * 2 b^3 /
wall time of the whole step.  Prints ONE JSON line.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_FP16_TFLOPS = 2500.0     # MI355X dense fp16 MFMA
PEAK_HBM_GBS = 8000.0         # MI355X HBM3E

PROFILE_DIR = os.path.join(ROOT, "profiles")

WORKLOADS = {
    # name: (N, tile, kind, lam, target kept ratio or None, fixed tau or None)
    # A target ratio that no tau > 0 reaches (after fp16 rounding the decay is exactly zero beyond a
    # short distance) gives the smallest positive norm product as tau: the largest kept fraction.
    "headline": (16384, 64, "exp", 0.003, 0.10, None),
    "headline_literal": (16384, 64, "exp", 0.1, 0.10, None),     # the decay rate as written: 10 % unreachable
    "headline_b32": (16384, 32, "exp", 0.003, 0.10, None),       # the reference's tile size (main.h:32 LoNum)
    "headline_b128": (16384, 128, "exp", 0.003, 0.10, None),
    "cfg2": (8192, 64, "exp", 0.01, 0.10, None),
    "cfg2_literal": (8192, 64, "exp", 0.1, 0.10, None),          # as written: 10 % unreachable
    "cfg3_05": (16384, 64, "alg", 0.0, 0.05, None),
    "cfg3_20": (16384, 64, "alg", 0.0, 0.20, None),
    "cfg3_max": (16384, 64, "alg", 0.0, 1.0, None),              # stands in for the unreachable 50 %
    "cfg4_dense": (16384, 64, "none", 0.0, None, 0.0),
    "cfg5": (65536, 128, "exp", 0.003, 0.02, None),
    "cfg5_literal": (65536, 128, "exp", 0.05, 0.02, None),       # as written: 2 % unreachable
    # the reference as checked out (para.h:1-14, cuSpAMM.cu:428-431): 2048^3, tile 32 (main.h:32), both operands
    # 0.1 / (|i-j|^0.1 + 1) with no random factor (getDecayMatrixAlg, tool.cu:426-436), Norm = 1.548969, and
    # fp16 inputs resident before the timed region (USINGHALF 1): the timed call is spamm_multiply_f16
    "ref_default": (2048, 32, "ref_alg", 0.0, None, 1.548969),
}
FP16_INPUT_WORKLOADS = ("ref_default",)


def paired_passes(N, tile, in_bytes, tau_aware):
    """Whether the library converts both operands of an N^3 multiply in one launch (normmap_pair_fits in
    kernels_normmap.hip): by tile rows of 1 KiB, at most 16384 of both together, 4096 if tau-aware.  The launch is
    reported as ms_normmap_b; tau-aware, it leaves out tiles of norm zero only, in both copies."""
    strips = 2 * (N // tile) * -(-N * int(in_bytes) // 1024)
    return strips <= (4096 if tau_aware else 16384)


def measured_traffic(workload, profile_dir=PROFILE_DIR):
    """HBM-side bytes per launch of each kernel of `workload`, read from the committed rocprofv3
    summaries: every profiles/*.txt carries lines `traffic <workload> <kernel key> <bytes>`
    (FETCH_SIZE and WRITE_SIZE per dispatch, each scaled by what the same counter reads for a
    plain device copy of known size).  Returns {key: bytes}; empty when no summary covers the
    workload -- the bench then reports traffic as null rather than a stale constant."""
    out = {}
    if not os.path.isdir(profile_dir):
        return out
    for name in sorted(os.listdir(profile_dir)):
        if not name.endswith(".txt"):
            continue
        for line in open(os.path.join(profile_dir, name)):
            f = line.split()
            if len(f) == 4 and f[0] == "traffic" and f[1] == workload:
                out[f[2]] = float(f[3])
    return out


def measured_trace_us(workload, profile_dir=PROFILE_DIR):
    """Average kernel duration in microseconds by `rocprofv3 --kernel-trace --stats`, from the lines
    `trace_us <workload> <kernel key> <microseconds>` of the committed summaries."""
    out = {}
    if not os.path.isdir(profile_dir):
        return out
    for name in sorted(os.listdir(profile_dir)):
        if not name.endswith(".txt"):
            continue
        for line in open(os.path.join(profile_dir, name)):
            f = line.split()
            if len(f) == 4 and f[0] == "trace_us" and f[1] == workload:
                out[f[2]] = float(f[3])
    return out


def gemm_structure(ctx, N, tile, kept, n_cu=256, cu_per_xcd=32):
    """Shape of the GEMM's work from the gate's own lists: how many macro tiles (256 x 256 of C) hold
    work, how they fall on the CUs, how much of the k loop runs kept-by-all ("full") stages, how
    full the others are, and how much of C is only zero-filled."""
    counts, sched = ctx.get_macro_counts()
    U, F = counts[..., 0].astype(np.int64), counts[..., 1].astype(np.int64)
    mt = 256 // tile                                  # output tiles per macro tile per dimension
    nspe = tile // 32                                 # 32-k stages per list entry
    computing = int((U > 0).sum())
    n_xcd = max(1, n_cu // cu_per_xcd)
    per_xcd = [int(v) for v in sched[:n_xcd]]
    stages, full_stages = int(U.sum()) * nspe, int(F.sum()) * nspe
    partial_entries = int((U - F).sum())
    kept_in_full = int(F.sum()) * mt * mt
    rounds_mean = computing / n_cu
    rounds_max = max(-(-v // cu_per_xcd) for v in per_xcd) if per_xcd else 0
    lens = U[U > 0]
    return {
        "macro_tiles": int(U.size), "computing_macro_tiles": computing, "empty_macro_tiles": int(U.size) - computing,
        "computing_per_xcd": per_xcd,
        "rounds_per_cu_mean": round(rounds_mean, 3), "rounds_per_cu_max": rounds_max,
        "round_quantisation_loss": round(1.0 - rounds_mean / rounds_max, 4) if rounds_max else None,
        "list_length_entries": {"mean": round(float(lens.mean()), 1) if lens.size else 0.0,
                                "min": int(lens.min()) if lens.size else 0, "max": int(lens.max()) if lens.size else 0},
        "stages": stages, "full_stage_share": round(full_stages / stages, 4) if stages else None,
        "partial_stage_share": round(1.0 - full_stages / stages, 4) if stages else None,
        "partial_stage_fill": (round((kept - kept_in_full) / (partial_entries * mt * mt), 4) if partial_entries else None),
        "zero_fill_bytes": (int(U.size) - computing) * 256 * 256 * 4,
        "zero_fill_share_of_c": round(1.0 - computing / U.size, 4),
    }


def decay_table(kind, n, lam):
    d = np.arange(n, dtype=np.float64)
    if kind == "exp":
        t = np.exp(-lam * d)
    elif kind == "alg":
        t = 1.0 / (1.0 + d) ** 2
    elif kind == "ref_alg":                 # c / (d^v + 1), c = v = 0.1, evaluated as the reference does (float pow)
        t = np.float32(0.1) / (np.power(d, np.float64(np.float32(0.1))).astype(np.float32) + np.float32(1))
    else:
        t = np.ones(n)
    return np.ascontiguousarray(t, dtype=np.float32)


def cpu_baseline(A, B, tile, tau, budget_s):
    """The host checker timed on a bounded sample of the same workload: full conversion,
    norm maps and gate, gated GEMM on as many leading tile rows as fit the time budget."""
    from oracle import oracle as orc
    threads = orc.num_threads()
    N = A.shape[0]
    nb = N // tile
    t0 = time.perf_counter()
    hA, hB = orc.f32_to_f16_bits(A), orc.f32_to_f16_bits(B)
    nA, nB = orc.normmap(hA, tile, 0), orc.normmap(hB, tile, 1)
    kept, counts, klist, mask = orc.gate(nA, nB, tau)
    Af, Bf = orc.f16_bits_to_f32(hA), orc.f16_bits_to_f32(hB)
    t_front = time.perf_counter() - t0
    C = np.zeros((N, N), dtype=np.float32)
    rows_done, prod_done, t_gemm = 0, 0, 0.0
    step = 2
    mid = nb // 2                      # start in the middle of the band: representative rows
    order = [mid]
    for d in range(1, nb):
        if mid + d < nb:
            order.append(mid + d)
        if mid - d >= 0:
            order.append(mid - d)
    i = 0
    while i < len(order) and t_gemm < budget_s:
        rows = order[i:i + step]
        t1 = time.perf_counter()
        for r in rows:
            orc.gemm_gated(Af, Bf, tile, counts, klist, ti0=r, ti1=r + 1, out=C)
        t_gemm += time.perf_counter() - t1
        rows_done += len(rows)
        prod_done += int(counts[rows].sum())
        i += step
    flops = prod_done * 2.0 * tile ** 3
    # whole-pipeline rate on the sample: front end scaled to the sampled share of rows
    t_total = t_gemm + t_front * rows_done / nb
    return dict(value=flops / t_total / 1e12 if t_total > 0 else 0.0, unit="TFLOP/s",
                cores=threads, kind="port",
                sample="%d of %d tile rows of the same workload (%d kept products): fp16 conversion, norm maps, "
                       "gate and gated GEMM of the host checker, %.1f s" % (rows_done, nb, prod_done, t_total),
                gemm_only_tflops=flops / t_gemm / 1e12 if t_gemm > 0 else 0.0,
                seconds=t_total), dict(C=C, rows=order[:rows_done], counts=counts, mask=mask, nA=nA, nB=nB,
                                       Af=Af, Bf=Bf, kept=kept)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--workload", default="headline", choices=sorted(WORKLOADS))
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--skip-literal", action="store_true", help="skip the one-off run of the literal lam=0.1 config")
    ap.add_argument("--skip-dense", action="store_true", help="skip the dense fp16 GEMM comparison")
    ap.add_argument("--no-prune", action="store_true",
                    help="timed multiplies without SPAMM_FLAG_PRUNE (the A pass then writes every fp16 tile)")
    ap.add_argument("--cpu-budget", type=float, default=12.0, help="seconds of host GEMM in the CPU sample")
    ap.add_argument("--skip-extras", action="store_true",
                    help="only the timed multiplies (profiling runs): no ceiling probe, tau = 0 run, dense GEMM, "
                         "error report, literal config or CPU baseline")
    ap.add_argument("--skip-variants", action="store_true",
                    help="skip the fp16-input / REUSE_B / A_EQ_B / no-prune timings")
    ap.add_argument("--calibrate-cache", action="store_true",
                    help="only run the read-only reference kernels of the dev library: 4 GiB streamed from HBM and a 96 MiB "
                         "buffer re-read from the memory-side cache, each with a full grid and with 32 workgroups: "
                         "reference points for the L2-miss read latency (TCC_EA0_RDREQ_LEVEL / TCC_EA0_RDREQ)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="only run a plain 1 GiB device copy 5 times (reference point for FETCH_SIZE/WRITE_SIZE)")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this build is single-GPU by design (the SpAMM path runs on one MI355X); "
              "run with --gpus 1", file=sys.stderr)
        sys.exit(2)

    import torch
    import cuspamm_amd as sp
    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        sys.exit(1)

    if args.calibrate_copy:
        x = torch.empty(1 << 28, dtype=torch.float32, device="cuda").normal_()
        y = torch.empty_like(x)
        for _ in range(5):
            y.copy_(x)
        torch.cuda.synchronize()
        print(json.dumps({"calibrate_copy_bytes_read": x.numel() * 4, "bytes_written": x.numel() * 4, "launches": 5}))
        return

    if args.calibrate_cache:
        from cuspamm_amd import dev as spdev
        names = ("hbm_stream_full_grid", "cache_reread_full_grid", "hbm_stream_32_workgroups", "cache_reread_32_workgroups")
        print(json.dumps({"calibrate_cache_GBps": {n: round(spdev.read_reference(0, i), 1) for i, n in enumerate(names)}}))
        return

    if args.skip_extras:
        args.no_cpu_baseline = args.skip_literal = args.skip_dense = args.skip_variants = True
    N, tile, kind, lam, ratio, tau = WORKLOADS[args.workload]
    nb = N // tile
    traffic = measured_traffic(args.workload)
    ctx = sp.SpammContext(0)          # runs on torch's current stream
    tab = decay_table(kind, N, lam)
    dA = torch.empty((N, N), dtype=torch.float32, device="cuda")
    dB = torch.empty((N, N), dtype=torch.float32, device="cuda")
    det = kind == "ref_alg"                     # the reference's generators carry no random factor
    ctx.fill_decay(dA, tab, 1, random=not det)
    ctx.fill_decay(dB, tab, 2, random=not det)
    dC = torch.empty((N, N), dtype=torch.float32, device="cuda")
    in16 = args.workload in FP16_INPUT_WORKLOADS
    # operands of the timed call: the fp32 matrices, or (the reference's own timed region, para.h:1,
    # cuSpAMM.cu:461-541) fp16 copies made before it
    tA, tB = (dA.half(), dB.half()) if in16 else (dA, dB)

    if tau is None:
        # fixed before the timed region: exact order statistic over the norm products, on the device
        ctx.normmap_f32(sp.ROLE_B, dB, tile)
        ctx.normmap_f32(sp.ROLE_A, dA, tile)
        tau, achieved = ctx.tau_for_ratio(ratio)
    else:
        achieved = None

    # the timed steps run the path as a caller would (no per-stage events between the kernels).
    # tau is an argument of the call, so the A pass (second, as in the reference) can leave out
    # the fp16 copy of tiles that no product keeps: same C, mask and counts, fewer bytes written.
    prune = not args.no_prune

    def wall_ms(call, steps, warmup):
        for _ in range(warmup):
            call()
        torch.cuda.synchronize()
        t_0 = time.perf_counter()
        for _ in range(steps):
            call()
        torch.cuda.synchronize()
        return (time.perf_counter() - t_0) * 1e3 / steps

    def event_ms(call, steps):
        acc = np.zeros(5)
        for _ in range(steps):
            call()
            s_ = ctx.get_stats()
            acc += [s_.ms_normmap_b, s_.ms_normmap_a, s_.ms_gate, s_.ms_gemm, s_.ms_total]
        return acc / steps, s_

    stage = np.zeros(5)
    ms_step = wall_ms(lambda: ctx.multiply(tA, tB, tile, tau, C=dC, prune=prune), args.steps, args.warmup)
    # per-kernel durations: HIP events recorded by the library on the stream the kernels run on;
    # re-run the same steps reading the events after each one (reading needs a sync, so it is
    # kept out of the wall-clock loop above)
    stage, st = event_ms(lambda: ctx.multiply(tA, tB, tile, tau, C=dC, timing=True, prune=prune), args.steps)
    # bytes the A pass writes: tile (i, k) is copied iff fl32(nA[i,k] * max_j nB[k,j]) >= tau; converted together
    # with B, every tile of non-zero norm
    nA_h, nB_h = ctx.get_normmap(sp.ROLE_A), ctx.get_normmap(sp.ROLE_B)
    # and the B pass every tile of non-zero norm
    a_tiles = nb * nb
    pruned = prune and tau > 0
    paired = paired_passes(N, tile, 2 if in16 else 4, pruned)

    def a_tiles_written(in_bytes):
        if not pruned:
            return a_tiles
        if paired_passes(N, tile, in_bytes, True):
            return int(np.count_nonzero(nA_h))
        return int(np.count_nonzero(nA_h * nB_h.max(axis=1)[None, :] >= np.float32(tau)))
    a_written = a_tiles_written(2 if in16 else 4)
    b_written = int(np.count_nonzero(nB_h)) if pruned else a_tiles
    kept, total = int(st.kept_products), int(st.total_products)
    flops = kept * 2.0 * tile ** 3
    value = flops / (ms_step * 1e-3) / 1e12
    gemm_tflops = flops / (stage[3] * 1e-3) / 1e12
    in_b = 2.0 if in16 else 4.0                                         # bytes per input element
    nm_bytes_all = in_b * N * N + 2.0 * N * N + 4.0 * nb * nb           # per matrix, every tile written
    nm_bytes_a = in_b * N * N + 2.0 * tile * tile * a_written + 4.0 * nb * nb
    nm_bytes_b = in_b * N * N + 2.0 * tile * tile * b_written + 8.0 * nb * nb
    # operand bytes the GEMM must read at least once: the distinct fp16 tiles A(i,k) / B(k,j) that some
    # kept product uses (from the gate's own bitmap), plus C written once
    gm = ctx.get_mask()                                                 # [nbM, nbN, words] uint64, bit k
    a_need = np.bitwise_or.reduce(gm, axis=1)                           # [nbM, words]: k tiles row i needs
    b_need = np.bitwise_or.reduce(gm, axis=0)                           # [nbN, words]
    a_tiles_read = int(np.unpackbits(a_need.view(np.uint8)).sum())
    b_tiles_read = int(np.unpackbits(b_need.view(np.uint8)).sum())
    del gm
    gemm_alg_bytes = 4.0 * N * N + 2.0 * tile * tile * (a_tiles_read + b_tiles_read)
    structure = gemm_structure(ctx, N, tile, kept)
    trace_us = measured_trace_us(args.workload)
    # the B pass; paired, the one launch, which also covers A's bytes
    nm_bytes = nm_bytes_b + (nm_bytes_a if paired else 0.0)
    nm_gbs = nm_bytes / (stage[0] * 1e-3) / 1e9
    nm_trace_us = trace_us.get("k_normmap_b", 0.0) + (trace_us.get("k_normmap_a", 0.0) if paired else 0.0)

    out = {
        "metric": "spamm_effective_tflops_kept_tiles",
        "value": round(value, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f16",
        "data": "synthetic",
        "config": {
            "workload": "N=%d tile=%d %s decay lam=%g seeded u_ij*decay(|i-j|), fp32 in HBM -> fp16 MFMA, fp32 C; "
                        "fixed tau=%.6e keeps %.2f%% of tile products" % (N, tile, kind, lam, tau, 100.0 * kept / total),
            "name": args.workload, "N": N, "tile": tile, "tau": tau, "target_kept_fraction": ratio,
            "kept_products": kept, "total_products": total,
            "kept_fraction": round(kept / total, 5),
            "prune": prune, "inputs": "fp16" if in16 else "fp32",
        },
        "stage_ms": {"normmap_b": round(stage[0], 4), "normmap_a": round(stage[1], 4), "gate": round(stage[2], 4),
                     "gemm": round(stage[3], 4), "sum_events": round(stage[4], 4)},
        "gemm_structure": structure,
        "gemm_only_tflops": round(gemm_tflops, 2),
        "gemm_only_frac_of_fp16_peak": round(gemm_tflops / PEAK_FP16_TFLOPS, 4),
        "whole_multiply_frac_of_fp16_peak": round(value / PEAK_FP16_TFLOPS, 4),
        "roofline": {
            "kernel": "k_gemm<%d> (gated MFMA GEMM)" % tile, "bound": "mfma",
            "achieved": round(gemm_tflops, 2), "peak": PEAK_FP16_TFLOPS, "unit": "TFLOP/s",
            "frac": round(gemm_tflops / PEAK_FP16_TFLOPS, 4),
            "traffic": traffic.get("k_gemm"),
            "flops_per_launch": flops, "avg_launch_ms": round(stage[3], 4),
            "frac_basis": "HIP events recorded by the library around the kernel on its stream, this run",
            "frac_by_kernel_trace": (round(flops / (trace_us["k_gemm"] * 1e-6) / 1e12 / PEAK_FP16_TFLOPS, 4)
                                     if "k_gemm" in trace_us else None),
            "kernel_trace_avg_launch_ms": round(trace_us["k_gemm"] * 1e-3, 4) if "k_gemm" in trace_us else None,
            "kernel_trace_basis": "rocprofv3 --kernel-trace average of the committed profiles/ summary (another run, another box)",
            "algorithmic_bytes_per_launch": gemm_alg_bytes,
            "algorithmic_operand_tiles": {"a": a_tiles_read, "b": b_tiles_read, "tile_bytes": 2 * tile * tile},
            "traffic_over_algorithmic": (round(traffic["k_gemm"] / gemm_alg_bytes, 3) if "k_gemm" in traffic else None),
        },
        "roofline_normmap": {
            "kernel": ("k_normmap_pair<%d> (both operands: fp16 copies + tile norms)" if paired
                       else "k_normmap<%d, B role> (fp32->fp16 + tile norms)") % tile, "bound": "hbm",
            "achieved": round(nm_gbs, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
            "frac": round(nm_gbs / PEAK_HBM_GBS, 4),
            "traffic": ((traffic["k_normmap_a"] + traffic["k_normmap_b"] if "k_normmap_a" in traffic else None) if paired
                        else traffic.get("k_normmap_b" if pruned else "k_normmap_b_unpruned")),
            "bytes_per_launch": nm_bytes, "avg_launch_ms": round(stage[0], 4),
            "frac_basis": "HIP events: the first stage's interval includes the gap before its kernel starts",
            "frac_by_kernel_trace": (round(nm_bytes / (nm_trace_us * 1e-6) / 1e9 / PEAK_HBM_GBS, 4)
                                     if nm_trace_us and pruned else None),
            "kernel_trace_avg_launch_ms": round(nm_trace_us * 1e-3, 4) if nm_trace_us else None,
            "tiles_written": b_written, "tiles": a_tiles, "bytes_per_launch_all_tiles": nm_bytes_all * (2 if paired else 1),
            "a_pass": {"tiles_written": a_written, "tiles": a_tiles, "bytes_per_launch": nm_bytes_a,
                       "in_the_launch_above": True} if paired else {"tiles_written": a_written, "tiles": a_tiles, "bytes_per_launch": nm_bytes_a,
                       "avg_launch_ms": round(stage[1], 4),
                       "achieved": round(nm_bytes_a / (stage[1] * 1e-3) / 1e9, 1),
                       "frac": round(nm_bytes_a / (stage[1] * 1e-3) / 1e9 / PEAK_HBM_GBS, 4),
                       "frac_basis": "HIP events: the interval also covers k_rowmax (a few microseconds)",
                       "frac_by_kernel_trace": (round(nm_bytes_a / (trace_us["k_normmap_a"] * 1e-6) / 1e9 / PEAK_HBM_GBS, 4)
                                                if "k_normmap_a" in trace_us and pruned else None),
                       "traffic": traffic.get("k_normmap_a" if pruned else "k_normmap_a_unpruned")},
        },
    }

    # The same multiply under the library's other calling conventions, each timed like the headline
    # (wall clock over whole calls, then per-stage events), outside the headline's timed loop.
    if not args.skip_variants:
        vsteps, vwarm = max(5, args.steps // 2), max(2, args.warmup // 2)
        variants = {}

        def variant(name, what, call_plain, call_timed, in_bytes_elem=None, written=None):
            ms = wall_ms(call_plain, vsteps, vwarm)
            sg, s_ = event_ms(call_timed, vsteps)
            fl = s_.kept_products * 2.0 * tile ** 3
            v = {"what": what, "ms_per_step": round(ms, 4), "value_tflops": round(fl / (ms * 1e-3) / 1e12, 2),
                 "kept_products": int(s_.kept_products),
                 "stage_ms": {"normmap_b": round(sg[0], 4), "normmap_a": round(sg[1], 4), "gate": round(sg[2], 4),
                              "gemm": round(sg[3], 4)}}
            if in_bytes_elem is not None:
                bw, aw = written
                bb = in_bytes_elem * N * N + 2.0 * tile * tile * bw + 8.0 * nb * nb
                ba = in_bytes_elem * N * N + 2.0 * tile * tile * aw + 4.0 * nb * nb
                def rate(nbytes, ms_):
                    gbs = nbytes / (ms_ * 1e-3) / 1e9
                    return {"bytes_per_launch": nbytes, "GBps": round(gbs, 1), "frac_of_hbm_peak": round(gbs / PEAK_HBM_GBS, 4)}
                if paired_passes(N, tile, in_bytes_elem, pruned and name != "no_prune"):
                    v["normmap_both_passes"] = rate(bb + ba, sg[0])
                else:
                    v["normmap_b_pass"], v["normmap_a_pass"] = rate(bb, sg[0]), rate(ba, sg[1])
            variants[name] = v

        if prune:
            variant("no_prune", "the timed call without SPAMM_FLAG_PRUNE: both passes write every fp16 tile",
                    lambda: ctx.multiply(tA, tB, tile, tau, C=dC),
                    lambda: ctx.multiply(tA, tB, tile, tau, C=dC, timing=True), in_b, (a_tiles, a_tiles))
        if not in16:
            hA, hB = dA.half(), dB.half()
            variant("fp16_inputs", "spamm_multiply_f16 on fp16 copies made before the timed region (the reference's "
                    "own timed region: para.h:1, cuSpAMM.cu:461-541); passes read 2 bytes per element",
                    lambda: ctx.multiply(hA, hB, tile, tau, C=dC, prune=prune),
                    lambda: ctx.multiply(hA, hB, tile, tau, C=dC, timing=True, prune=prune), 2.0, (b_written, a_tiles_written(2)))
            del hA, hB
        # one B against many A: B's fp16 copy and norm map stay resident (A's pass, gate, GEMM remain)
        ctx.multiply(tA, tB, tile, tau, C=dC, prune=prune)
        variant("reuse_b", "SPAMM_FLAG_REUSE_B: B's fp16 copy and norm map kept from the previous call",
                lambda: ctx.multiply(tA, tB, tile, tau, C=dC, prune=prune, reuse_b=True),
                lambda: ctx.multiply(tA, tB, tile, tau, C=dC, timing=True, prune=prune, reuse_b=True))
        # A = B (BASELINE's first configuration, matrix powers): one read feeds both operand roles; the product
        # is A*A, so its kept count is its own
        variant("a_eq_b", "SPAMM_FLAG_A_EQ_B on A*A: one pass reads the matrix once and writes both packed copies "
                "(reported as normmap_b); beside it the same product as two passes",
                lambda: ctx.multiply(tA, tA, tile, tau, C=dC, prune=prune, a_eq_b=True),
                lambda: ctx.multiply(tA, tA, tile, tau, C=dC, timing=True, prune=prune, a_eq_b=True))
        variants["a_eq_b"]["two_pass_ms_per_step"] = round(
            wall_ms(lambda: ctx.multiply(tA, tA, tile, tau, C=dC, prune=prune), vsteps, vwarm), 4)
        out["variants"] = variants
        out["no_prune_ms_per_step"] = variants["no_prune"]["ms_per_step"] if "no_prune" in variants else round(ms_step, 4)

    # what the matrix pipeline sustains on this box with nothing but MFMAs: with random operands
    # the clock settles well below the datasheet's (power management), so this, not the datasheet
    # peak, is what a GEMM on real data can approach; and a dense fp16 GEMM of the same size by the
    # vendor library (the analogue of the reference's cuBLAS comparison, tool.cu:153-226)
    if not args.skip_extras:
        from cuspamm_amd import dev as spdev
        tf_rand, ghz_rand = spdev.mfma_ceiling(0, True)
        tf_zero, ghz_zero = spdev.mfma_ceiling(0, False)
        out["mfma_ceiling"] = {
            "random_operands_tflops": round(tf_rand, 1), "random_operands_clock_ghz": round(ghz_rand, 3),
            "zero_operands_tflops": round(tf_zero, 1), "zero_operands_clock_ghz": round(ghz_zero, 3),
            "gemm_frac_of_random_operand_ceiling": round(gemm_tflops / tf_rand, 4),
        }
    if not args.skip_dense and N <= 16384:
        hA, hB = dA.half(), dB.half()
        for _ in range(3):
            hC = torch.matmul(hA, hB)
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(5):
            hC = torch.matmul(hA, hB)
        e1.record()
        torch.cuda.synchronize()
        dense_ms = e0.elapsed_time(e1) / 5
        out["dense_fp16_gemm"] = {
            "library": "hipBLASLt via torch.matmul (fp16 in, fp16 out, conversion not timed)",
            "ms": round(dense_ms, 4), "tflops": round(2.0 * N ** 3 / (dense_ms * 1e-3) / 1e12, 1),
            "spamm_gemm_speedup": round(dense_ms / stage[3], 2),
            "spamm_whole_multiply_speedup": round(dense_ms / ms_step, 2),
        }
        del hA, hB, hC
        # the gated GEMM itself as a dense GEMM on the SAME matrices (tau = 0 keeps every product):
        # beside the vendor figure above it separates what the kernel loses from what the data and
        # the power limit cost both alike (decaying matrices are mostly tiny values: both run
        # faster on them than on uniform data)
        t0ms = []
        for _ in range(4):
            ctx.multiply(dA, dB, tile, 0.0, C=dC, timing=True)
            t0ms.append(ctx.get_stats().ms_gemm)
        t0 = float(np.median(t0ms[1:]))
        out["gemm_tau0_same_data"] = {
            "what": "k_gemm at tau = 0 (all %d^3 tile products) on the benchmark's own A and B" % nb,
            "ms": round(t0, 4), "tflops": round(2.0 * N ** 3 / (t0 * 1e-3) / 1e12, 1),
            "frac_of_fp16_peak": round(2.0 * N ** 3 / (t0 * 1e-3) / 1e12 / PEAK_FP16_TFLOPS, 4),
            "vs_vendor_dense_gemm_on_same_data": round(dense_ms / t0, 4),
        }

    # error against an exact fp64 dense product of the same fp16 operands, whole matrix, next to
    # the tau-derived bound (both formed on the device, outside the timed region)
    if N <= 16384 and not args.skip_extras:
        ctx.multiply(tA, tB, tile, tau, C=dC)
        e64, d64, c64 = ctx.error_vs_dense(dC)
        bound = ctx.dropped_bound(tau)
        # fp32 accumulation of K terms leaves ~eps32 * sqrt(K) relative noise on the kept part even
        # when nothing is dropped: a tau bound below that floor is not violated by an error above it
        floor = float(np.finfo(np.float32).eps) * np.sqrt(N) * d64
        out["error_vs_fp64_dense"] = {
            "frobenius_error": float("%.6e" % e64), "dense_frobenius": float("%.6e" % d64),
            "relative": float("%.3e" % (e64 / d64 if d64 else 0.0)),
            "tau_bound_frobenius": float("%.6e" % bound),
            "rounding_floor_frobenius": float("%.6e" % floor),
            "rounding_floor_is": "eps_fp32 * sqrt(K) * ||dense||_F (fp32 accumulation noise, present at tau = 0 too)",
            "within_bound_plus_floor": bool(e64 <= bound + floor),
            "rows": N,
        }

    if args.workload == "headline" and not args.skip_dense:
        # What a dense GEMM reaches on operands like the ones the kept products multiply.  45 % of
        # the headline's fp16 entries are exactly zero (the decay underflows beyond |i-j| ~ 5500),
        # and a dense product over them draws less power and runs at a higher clock than one over
        # non-zero values; the 10 % band multiplies entries within ~4000 of the diagonal only.  The
        # same decay folded to distances below 4096 everywhere gives both dense kernels operands
        # like the band's: the rate a gated GEMM on this band would reach with no structural loss.
        period = 4096
        tab_f = np.ascontiguousarray(tab[np.arange(N) % period])
        fA, fB = torch.empty_like(dA), torch.empty_like(dB)
        ctx.fill_decay(fA, tab_f, 1)
        ctx.fill_decay(fB, tab_f, 2)
        fms = []
        for _ in range(4):
            ctx.multiply(fA, fB, tile, 0.0, C=dC, timing=True)
            fms.append(ctx.get_stats().ms_gemm)
        f0 = float(np.median(fms[1:]))
        hA, hB = fA.half(), fB.half()
        zeros = float((hA == 0).float().mean())
        for _ in range(3):
            hC = torch.matmul(hA, hB)
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(5):
            hC = torch.matmul(hA, hB)
        e1.record()
        torch.cuda.synchronize()
        fv = e0.elapsed_time(e1) / 5
        ours_tf, vendor_tf = 2.0 * N ** 3 / (f0 * 1e-3) / 1e12, 2.0 * N ** 3 / (fv * 1e-3) / 1e12
        out["dense_rate_on_band_like_values"] = {
            "what": "dense fp16 GEMMs (k_gemm at tau = 0, hipBLASLt) on the same decay folded to |i-j| mod %d: "
                    "no zero entries, like the operands of the kept products" % period,
            "fp16_zero_entries": round(zeros, 4),
            "k_gemm_tau0_tflops": round(ours_tf, 1), "k_gemm_tau0_frac_of_fp16_peak": round(ours_tf / PEAK_FP16_TFLOPS, 4),
            "vendor_dense_tflops": round(vendor_tf, 1), "vendor_dense_frac_of_fp16_peak": round(vendor_tf / PEAK_FP16_TFLOPS, 4),
            "gated_gemm_vs_k_gemm_tau0": round(gemm_tflops / ours_tf, 4),
            "gated_gemm_vs_vendor_dense": round(gemm_tflops / vendor_tf, 4),
        }
        del fA, fB, hA, hB, hC

    if args.workload == "headline" and not args.skip_literal:
        # the decay rate as literally written in the config, run once for the record
        tab_l = decay_table("exp", N, 0.1)
        lA = torch.empty_like(dA)
        lB = torch.empty_like(dB)
        ctx.fill_decay(lA, tab_l, 1)
        ctx.fill_decay(lB, tab_l, 2)
        ctx.normmap_f32(sp.ROLE_B, lB, tile)
        ctx.normmap_f32(sp.ROLE_A, lA, tile)
        ltau, lach = ctx.tau_for_ratio(0.10)
        best = 1e9
        for _ in range(5):
            ctx.multiply(lA, lB, tile, ltau, C=dC, timing=True)
            lst = ctx.get_stats()
            best = min(best, lst.ms_total)
        out["literal_config"] = {
            "workload": "N=%d tile=%d exp decay lam=0.1 as written; 10%% kept is unreachable after fp16 rounding" % (N, tile),
            "tau": ltau, "kept_fraction": round(lst.kept_products / lst.total_products, 6),
            "ms_per_multiply": round(best, 4),
            "effective_tflops": round(lst.kept_products * 2.0 * tile ** 3 / (best * 1e-3) / 1e12, 2),
        }
        del lA, lB

    if not args.no_cpu_baseline and N <= 16384:
        A, B = dA.cpu().numpy(), dB.cpu().numpy()
        same_c = None
        if prune:
            plain = ctx.multiply(tA, tB, tile, tau).clone()
        ctx.multiply(tA, tB, tile, tau, C=dC, prune=prune)      # the call that was timed
        if prune:
            same_c = bool(torch.equal(plain, dC))
            del plain
        gmask = ctx.get_mask()
        base, chk = cpu_baseline(A, B, tile, tau, args.cpu_budget)
        out["cpu_baseline"] = {k: (round(v, 5) if isinstance(v, float) else v) for k, v in base.items()}
        # parity on the sample: bit-exact mask over the whole problem, C on the sampled rows
        from oracle import oracle as orc
        rows = chk["rows"]
        sel = np.concatenate([np.arange(r * tile, (r + 1) * tile) for r in rows])
        Cg = dC[torch.from_numpy(sel).cuda()].cpu().numpy()
        err, nrm, _ = orc.frob_diff(Cg, chk["C"][sel])
        d_err, d_nrm, bound = 0.0, 0.0, 0.0
        for r in rows[:2]:
            dense = orc.gemm_dense_f64(chk["Af"], chk["Bf"], r * tile, (r + 1) * tile)
            e, n_, _ = orc.frob_diff(dC[r * tile:(r + 1) * tile].cpu().numpy(), dense)
            d_err += e * e
            d_nrm += n_ * n_
            bound += orc.dropped_bound(chk["nA"], chk["nB"], tau, r, r + 1) ** 2
        out["parity"] = {
            "mask_bit_exact": bool(np.array_equal(gmask, chk["mask"])),
            "kept_products_match": bool(chk["kept"] == kept),
            "c_rel_frobenius_vs_checker": float("%.3e" % (err / nrm if nrm else 0.0)),
            "c_tolerance": 1e-3,
            "err_vs_fp64_dense_frobenius": float("%.4e" % np.sqrt(d_err)),
            "fp64_dense_frobenius": float("%.4e" % np.sqrt(d_nrm)),
            "tau_bound_frobenius": float("%.4e" % np.sqrt(bound)),
            "rounding_floor_frobenius": float("%.4e" % (float(np.finfo(np.float32).eps) * np.sqrt(N) * np.sqrt(d_nrm))),
            "rows_checked": len(rows), "rows_vs_fp64": 2,
            "prune_c_bit_identical_to_plain_call": same_c,
        }
    elif not args.no_cpu_baseline:
        out["cpu_baseline"] = None

    ctx.close()
    print(json.dumps(out))


if __name__ == "__main__":
    main()
