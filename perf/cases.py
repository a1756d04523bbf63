"""Cases by which the speed of the engine is measured: what a program that multiplies with it asks of it.

A case names one way of using the engine (`op`), the shape, the tile size, the input type, the values of the operands
and how much is kept.  `listed()` has the ones that stand for the configurations of bench.py and the tests, `draw()`
gives others of the same ranges.  Operands are fp32 or fp16 tensors on the GPU whose entries decay away from the
diagonal, u_ij * decay(|i - j|) with u_ij uniform in [-1, 1): the matrices the method is for; tau is the threshold that
keeps the wanted fraction of the tile products of exactly these operands.

    multiply   C = A B, as is
    prune      C = A B with the tau-aware conversion passes
    noalloc    C = A B in the library's fixed workspace (no device allocation)
    reuse_b    a new A against a B that was converted before
    square     A A, the matrix read once for both roles
    to_ratio   tau found for a kept fraction (order statistic), then gate and multiply
    tuned      tau found by the reference's bisection, then gate and multiply
    report     error against the exact product and the tau-derived bounds of a finished multiply
"""
import math

import torch

import cuspamm_amd as sp

DEVICE = 0
_stream = None


def _program_stream():
    """The one stream a program issues its multiplies on (calls in the fixed workspace must not overlap)."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream(DEVICE)
    return _stream


def _case(name, op, M, K, N, tile, decay, rate, keep, dtype="fp32", row0=0):
    c = {"op": op, "M": M, "K": K, "N": N, "tile": tile, "decay": decay, "rate": rate, "keep": keep, "dtype": dtype, "row0": row0}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one small block of a larger program: all launches and latency
        _case("block_256_t32", "multiply", 256, 256, 256, 32, "exp", 0.1, 0.2),
        # a serving step under a no-allocation rule; no dimension is a multiple of the 256-wide work units
        _case("serving_ragged_t32", "noalloc", 1056, 1568, 1312, 32, "exp", 0.02, 0.15),
        # the reference's default experiment: its size, tile, decay family and input type, at the fraction its tau keeps
        _case("reference_default_t32_fp16", "multiply", 2048, 2048, 2048, 32, "ref", 0.1, 0.05, "fp16"),
        # the same with the reference's tuner in front, as its timed loop has it (75 % +- 1 %, at most 20 rounds)
        _case("reference_tuned_t32_fp16", "tuned", 2048, 2048, 2048, 32, "ref", 0.1, 0.75, "fp16"),
        # a rectangular problem whose tau is chosen by the kept fraction
        _case("rectangular_to_ratio_t32", "to_ratio", 5024, 4128, 3168, 32, "alg", 2.0, 0.10),
        # slabs of rows streamed against a resident B
        _case("row_slab_reuse_b_t64", "reuse_b", 1024, 8192, 8192, 64, "exp", 0.01, 0.05, row0=3584),
        # a step of a matrix power
        _case("square_8192_t64", "square", 8192, 8192, 8192, 64, "exp", 0.01, 0.10),
        # nothing dropped: the engine as a plain GEMM
        _case("dense_8192_t64", "multiply", 8192, 8192, 8192, 64, "none", 0.0, 1.0),
        # slow algebraic decay, fp16-resident operands, ragged at the work units
        _case("algebraic_10048_t64_fp16", "multiply", 10048, 10048, 10048, 64, "alg", 2.0, 0.20, "fp16"),
        # the headline workload
        _case("band_16384_t64", "prune", 16384, 16384, 16384, 64, "exp", 0.003, 0.10),
        # the largest: a narrow band at the widest tile, mostly passes over the operands and zeros of C
        _case("band_32768_t128", "prune", 32768, 32768, 32768, 128, "exp", 0.003, 0.02),
        # accuracy of a finished multiply
        _case("error_report_4096_t64", "report", 4096, 4096, 4096, 64, "exp", 0.01, 0.05),
    ]


# largest side by use; the smallest is one or a few tiles
_SIDES = {"multiply": 20000, "prune": 20000, "noalloc": 2200, "reuse_b": 12000, "square": 16000, "to_ratio": 8000,
          "tuned": 4000, "report": 4096}
_MAX_FLOPS = 1.3e12
_MAX_BYTES = 12.0e9


def _side(rng, tile, top):
    low = max(256, tile)
    v = math.exp(rng.uniform(math.log(low), math.log(top)))
    return max(1, int(v / tile + 0.5)) * tile


def draw(rng):
    op = rng.choice(["multiply", "multiply", "prune", "prune", "noalloc", "reuse_b", "square", "to_ratio", "tuned", "report"])
    tile = rng.choice([32, 64, 128])
    dtype = "fp32" if op in ("noalloc", "reuse_b") else rng.choice(["fp32", "fp32", "fp16"])
    top = _SIDES[op]
    M, K, N = (_side(rng, tile, top) for _ in range(3))
    if op == "square" or (op in ("multiply", "prune") and rng.random() < 0.5):
        K = N = M
    if op == "reuse_b":
        M = _side(rng, tile, top // 8)
    if op == "report":
        unit = max(64, tile)
        M, K, N = (max(1, x // unit) * unit for x in (M, K, N))
    decay = rng.choice(["exp", "exp", "alg", "ref", "none"])
    long = max(M, K, N)
    if decay == "exp":
        rate = round(rng.uniform(20.0, 60.0) / long, 6)
        keep = math.exp(rng.uniform(math.log(0.02), math.log(0.15)))
    elif decay == "alg":
        rate, keep = 2.0, math.exp(rng.uniform(math.log(0.02), math.log(0.30)))
    elif decay == "ref":
        rate, keep = 0.1, math.exp(rng.uniform(math.log(0.02), math.log(0.50)))
    else:
        rate, keep = 0.0, 1.0 if op in ("multiply", "noalloc", "square") else 0.5
    if op == "tuned":
        decay, rate, keep = rng.choice([("ref", 0.1), ("alg", 2.0)]) + (rng.choice([0.25, 0.5, 0.75]),)
    flops = 2.0 * M * K * N
    if keep < 1.0:
        keep = round(min(keep, _MAX_FLOPS / flops), 6)
    elif flops > _MAX_FLOPS:
        keep = round(_MAX_FLOPS / flops, 6)
    c = _case(None, op, M, K, N, tile, decay, rate, keep, dtype)
    if op == "reuse_b" and K > M:
        c["row0"] = rng.randrange(0, K - M + 1, tile)
    return c


def _operand(rows, cols, case, seed, row0=0):
    """u_ij * decay(|row0 + i - j|) with u_ij uniform in [-1, 1), fp32 or fp16, made in slabs of rows."""
    d = torch.arange(row0 + max(rows, cols) + 1, dtype=torch.float64, device="cuda")
    kind, rate = case["decay"], case["rate"]
    if kind == "exp":
        table = torch.exp(-rate * d)
    elif kind == "alg":
        table = (1.0 + d) ** -rate
    elif kind == "ref":
        table = 0.1 / (d ** rate + 1.0)
    else:
        table = torch.ones_like(d)
    table = table.float()
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    half = case["dtype"] == "fp16"
    X = torch.empty((rows, cols), dtype=torch.float16 if half else torch.float32, device="cuda")
    j = torch.arange(cols, device="cuda")
    step = max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        i = torch.arange(row0 + r, row0 + min(r + step, rows), device="cuda")
        u = torch.rand((i.numel(), cols), generator=g, device="cuda") * 2.0 - 1.0
        X[r:r + step] = u * table[(i[:, None] - j[None, :]).abs()]
    return X


def prepare(case, seed):
    M, K, N, tile, op = case["M"], case["K"], case["N"], case["tile"], case["op"]
    A = _operand(M, K, case, 2 * seed + 1, case["row0"])
    B = A if op == "square" else _operand(K, N, case, 2 * seed + 2)
    C = torch.empty((M, N), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(_program_stream()):
        ctx = sp.SpammContext(DEVICE)
    normmap = ctx.normmap_f16 if case["dtype"] == "fp16" else ctx.normmap_f32
    tau = 0.0
    if case["keep"] < 1.0 and op not in ("to_ratio", "tuned"):
        normmap(sp.ROLE_B, B, tile)
        normmap(sp.ROLE_A, A, tile)
        tau = ctx.tau_for_ratio(case["keep"])[0]
    elif op == "reuse_b":
        normmap(sp.ROLE_B, B, tile)
    if op == "report":
        ctx.multiply(A, B, tile, tau, C)
    return {"case": case, "ctx": ctx, "A": A, "B": B, "C": C, "tau": tau, "normmap": normmap}


def run(state):
    case, ctx, A, B, C, tau = (state[k] for k in ("case", "ctx", "A", "B", "C", "tau"))
    op, tile = case["op"], case["tile"]
    if op == "multiply":
        return ctx.multiply(A, B, tile, tau, C)
    if op == "prune":
        return ctx.multiply(A, B, tile, tau, C, prune=True)
    if op == "noalloc":
        return ctx.multiply_noalloc(A, B, tile, tau, C)
    if op == "reuse_b":
        return ctx.multiply(A, B, tile, tau, C, reuse_b=True)
    if op == "square":
        return ctx.multiply(A, B, tile, tau, C, a_eq_b=True)
    if op == "report":
        return ctx.error_vs_dense(C), ctx.dropped_bound(tau), ctx.dropped_bound_tiles(tau)
    state["normmap"](sp.ROLE_B, B, tile)
    state["normmap"](sp.ROLE_A, A, tile)
    if op == "to_ratio":
        found = ctx.tau_for_ratio(case["keep"])
    else:
        found = ctx.tune_bisect(case["keep"], 0.01, 20)
    ctx.gate(found[0])
    return ctx.gemm_gated(C), found


def work(case):
    """Operands read once and C written once; two operations per kept multiply-add (all of them in the report)."""
    M, K, N, tile, op = case["M"], case["K"], case["N"], case["tile"], case["op"]
    e = 2 if case["dtype"] == "fp16" else 4
    flops = 2.0 * M * K * N * case["keep"]
    if op == "report":         # the engine's fp16 copies and C are read, one bound per output tile is written
        return {"bytes": 2 * (M * K + K * N) + 4 * M * N + 8 * (M // tile) * (N // tile), "flops": 2.0 * M * K * N}
    operands = M * K if op == "square" else M * K + K * N
    if op == "reuse_b":        # B lies there as fp16
        return {"bytes": e * M * K + 2 * K * N + 4 * M * N, "flops": flops}
    return {"bytes": e * operands + 4 * M * N, "flops": flops}


def tolerance(case):
    # the kept products of these cases summed in the opposite order of k: at most 7.5e-7 (2-norm) and 9e-6 of the
    # result's root mean square (dense and band, K = 8192); against 64-bit sums no more; tau is an exact order statistic
    return {"rel": 4e-6, "max": 4e-5}
