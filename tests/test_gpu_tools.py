"""fp16-input entry point, operand reuse and the error-report tooling."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _vs_checker(orc, ctx, C, A32, B32, tile, tau, what):
    """The library's last multiply against the host checker run on the same fp32 values: kept mask,
    counts and norm maps bit-exact, C within 1e-3 relative Frobenius error."""
    ref = orc.spamm(np.ascontiguousarray(A32, dtype=np.float32), np.ascontiguousarray(B32, dtype=np.float32), tile, tau)
    assert np.array_equal(ctx.get_mask(), ref["mask"]), what
    assert np.array_equal(ctx.get_counts(), ref["counts"]), what
    assert np.array_equal(ctx.get_normmap(0).view(np.uint32), ref["nA"].view(np.uint32)), what
    assert np.array_equal(ctx.get_normmap(1).view(np.uint32), ref["nB"].view(np.uint32)), what
    assert ctx.get_stats().kept_products == ref["kept"], what
    err, nrm, _ = orc.frob_diff(C.cpu().numpy(), ref["C"])
    assert err <= 1e-3 * nrm, "%s: C off by %g" % (what, err / max(nrm, 1e-300))
    return ref


@pytest.mark.parametrize("tile", [32, 64, 128])
def test_fp16_inputs_equal_fp32_inputs_of_the_same_values(orc, ctx, tile):
    import torch
    M, K, N = 3 * 128, 2 * 128, 4 * 128
    tab = orc.decay_table("exp", max(M, K, N), 0.01)
    A = _dev(orc.fill_decay(M, K, tab, 1)).half()
    B = _dev(orc.fill_decay(K, N, tab, 2)).half()
    ctx.normmap_f16(1, B, tile)
    ctx.normmap_f16(0, A, tile)
    tau, ach = ctx.tau_for_ratio(0.5)
    assert 0.45 < ach < 0.6
    C16 = ctx.multiply(A, B, tile, tau).clone()
    # fp16 is the reference's real input type (para.h:1, cuSpAMM.cu:486): the checker, fed the same
    # values as fp32 (its fp16 rounding is then the identity), must agree
    _vs_checker(orc, ctx, C16, A.float().cpu().numpy(), B.float().cpu().numpy(), tile, tau, "fp16 inputs")
    m16, nA16, nB16 = ctx.get_mask(), ctx.get_normmap(0), ctx.get_normmap(1)
    assert np.array_equal(ctx.get_fp16(0), A.cpu().numpy().view(np.uint16))
    assert np.array_equal(ctx.get_fp16(1), B.cpu().numpy().view(np.uint16))
    C32 = ctx.multiply(A.float(), B.float(), tile, tau)
    assert np.array_equal(ctx.get_mask(), m16)
    assert np.array_equal(ctx.get_normmap(0).view(np.uint32), nA16.view(np.uint32))
    assert np.array_equal(ctx.get_normmap(1).view(np.uint32), nB16.view(np.uint32))
    assert torch.equal(C16, C32)
    Cp = ctx.multiply(A, B, tile, tau, prune=True)      # tau-aware passes on fp16 inputs
    assert torch.equal(C16, Cp)
    _vs_checker(orc, ctx, Cp, A.float().cpu().numpy(), B.float().cpu().numpy(), tile, tau, "fp16 inputs, tau-aware")
    kept = ctx.get_stats().kept_products
    assert 0 < kept < (M // tile) * (K // tile) * (N // tile)


def test_operand_reuse(orc, ctx):
    import torch
    import cuspamm_amd as sp
    n = 512
    tab = orc.decay_table("exp", n, 0.01)
    A1, A2, B = (_dev(orc.fill_decay(n, n, tab, s)) for s in (1, 3, 2))
    ref1 = ctx.multiply(A1, B, 64, 0.5).clone()
    ref2 = ctx.multiply(A2, B, 64, 0.5).clone()
    ctx.multiply(A1, B, 64, 0.5)
    hA1, hA2, hB = A1.cpu().numpy(), A2.cpu().numpy(), B.cpu().numpy()
    got2 = ctx.multiply(A2, B, 64, 0.5, reuse_b=True)          # B's fp16 copy and norm map are kept
    assert torch.equal(got2, ref2)
    _vs_checker(orc, ctx, got2, hA2, hB, 64, 0.5, "new A against the resident B")
    got1 = ctx.multiply(A1, B, 64, 0.5, reuse_b=True)
    assert torch.equal(got1, ref1)
    _vs_checker(orc, ctx, got1, hA1, hB, 64, 0.5, "first A again against the resident B")
    got1 = ctx.multiply(A1, B, 64, 0.1, reuse_a=True, reuse_b=True)   # only tau changes
    _vs_checker(orc, ctx, got1, hA1, hB, 64, 0.1, "both operands resident, new tau")
    assert torch.equal(got1.clone(), ctx.multiply(A1, B, 64, 0.1))
    # a new B against the resident A (matrix powers: X, then X * B2)
    B2 = _dev(orc.fill_decay(n, n, tab, 9))
    ctx.multiply(A1, B, 64, 0.5)
    gotb = ctx.multiply(A1, B2, 64, 0.5, reuse_a=True)
    _vs_checker(orc, ctx, gotb, hA1, B2.cpu().numpy(), 64, 0.5, "new B against the resident A")
    with pytest.raises(sp.SpammError) as ei:                    # shape changed: nothing to reuse
        ctx.multiply(A1[:256].contiguous(), B, 64, 0.5, reuse_a=True)
    assert ei.value.code == -4


def test_error_report_matches_checker(orc, ctx):
    n, tile = 512, 64
    tab = orc.decay_table("exp", n, 0.01)
    A, B = orc.fill_decay(n, n, tab, 1), orc.fill_decay(n, n, tab, 2)
    for tau in (0.0, 0.5, 3.0):
        C = ctx.multiply(_dev(A), _dev(B), tile, tau)
        Af = orc.f16_bits_to_f32(ctx.get_fp16(0))
        Bf = orc.f16_bits_to_f32(ctx.get_fp16(1))
        dense = orc.gemm_dense_f64(Af, Bf)
        e, d, c = orc.frob_diff(C.cpu().numpy(), dense)
        ge, gd, gc = ctx.error_vs_dense(C)
        assert abs(gd - d) <= 1e-10 * d and abs(gc - c) <= 1e-10 * c
        assert abs(ge - e) <= 1e-6 * e + 1e-12 * d
        bound = orc.dropped_bound(ctx.get_normmap(0), ctx.get_normmap(1), tau)
        gb = ctx.dropped_bound(tau)
        assert abs(gb - bound) <= 1e-9 * max(bound, 1e-30)
        assert ge <= gb * (1 + 1e-4) + 1e-5 * gd
        # per output tile: the dropped sums themselves, against the checker's, and consistent with
        # the scalar (root of the sum of squares, whole matrix and a row range)
        gt = ctx.dropped_bound_tiles(tau)
        ot = orc.dropped_bound_tiles(ctx.get_normmap(0), ctx.get_normmap(1), tau)
        assert gt.shape == ot.shape == (n // tile, n // tile)
        assert np.all(np.abs(gt - ot) <= 1e-12 * np.maximum(ot, 1e-300)), np.abs(gt - ot).max()
        assert np.array_equal(gt == 0, ot == 0)
        assert abs(np.sqrt((gt ** 2).sum()) - gb) <= 1e-9 * max(gb, 1e-30)
        part = orc.dropped_bound(ctx.get_normmap(0), ctx.get_normmap(1), tau, 2, 5)
        assert abs(np.sqrt((gt[2:5] ** 2).sum()) - part) <= 1e-9 * max(part, 1e-30)
        # row range
        ge2, gd2, _ = ctx.error_vs_dense(C, 128, 256)
        e2, d2, _ = orc.frob_diff(C.cpu().numpy()[128:256], dense[128:256])
        assert abs(gd2 - d2) <= 1e-10 * d2 and abs(ge2 - e2) <= 1e-6 * e2 + 1e-12 * d2


@pytest.mark.parametrize("tile", [32, 64, 128])
def test_a_equals_b_single_pass(orc, ctx, tile):
    # BASELINE config 1 shape (A = B): one read of the matrix must give the same fp16 copies, norm
    # maps, mask and C as the two-pass run
    import torch
    import cuspamm_amd as sp
    n = 1024
    tab = orc.decay_table("exp", n, 0.5 if tile == 32 else 0.05)
    X = _dev(orc.fill_decay(n, n, tab, 1))
    tau = 1e-4 if tile == 32 else 2.0
    C2 = ctx.multiply(X, X, tile, tau).clone()
    ref = (ctx.get_mask(), ctx.get_normmap(0), ctx.get_normmap(1), ctx.get_fp16(0), ctx.get_fp16(1))
    C1 = ctx.multiply(X, X, tile, tau, a_eq_b=True)
    hX = X.cpu().numpy()
    chk = _vs_checker(orc, ctx, C1, hX, hX, tile, tau, "A = B single pass")
    assert np.array_equal(ctx.get_fp16(0), chk["hA"]) and np.array_equal(ctx.get_fp16(1), chk["hB"])
    got = (ctx.get_mask(), ctx.get_normmap(0), ctx.get_normmap(1), ctx.get_fp16(0), ctx.get_fp16(1))
    for r, g in zip(ref, got):
        assert np.array_equal(r.view(np.uint8), g.view(np.uint8))
    assert torch.equal(C1, C2)
    kept = ctx.get_stats().kept_products
    assert 0 < kept < (n // tile) ** 3
    with pytest.raises(sp.SpammError):                       # the flag needs the same pointer and a square problem
        ctx.multiply(X, X.clone(), tile, tau, a_eq_b=True)
    # the single pass with the tau-aware flag: tiles of norm zero are left out of both copies
    # (exp(-0.5 d) is exactly zero in fp16 beyond d = 33, exp(-0.05 d) beyond d = 333)
    assert np.count_nonzero(ref[1] == 0) > 0
    ctx.multiply(torch.full_like(X, 1000.0), X, tile, 0.0)   # loud workspace
    Cp = ctx.multiply(X, X, tile, tau, a_eq_b=True, prune=True)
    assert torch.equal(Cp, C2)
    assert np.array_equal(ctx.get_mask(), ref[0])
    _vs_checker(orc, ctx, Cp, hX, hX, tile, tau, "A = B single pass, tau-aware")
    with pytest.raises(sp.SpammError):
        ctx.get_fp16(0)
    with pytest.raises(sp.SpammError):
        ctx.get_fp16(1)
    assert torch.equal(ctx.multiply(X, X, tile, tau * 3, reuse_a=True, reuse_b=True), ctx.multiply(X, X, tile, tau * 3))


@pytest.mark.parametrize("tile", [32, 64, 128])
def test_tau_aware_passes_give_the_same_product(orc, ctx, tile):
    """SPAMM_FLAG_PRUNE: tiles that no product can keep are not copied -- at this size, where one launch converts
    both operands, those of norm zero in either (the A pass of its own, which knows B's norms, has a test below);
    C, mask, counts and norm maps must not change.  The workspace is first filled with loud
    operands so that a GEMM reading a skipped tile would show."""
    import torch
    import cuspamm_amd as sp
    M, K, N = 4 * 256, 3 * 256, 2 * 256 + tile
    tab = orc.decay_table("exp", max(M, K, N), 0.05)      # exactly zero in fp16 beyond |i - j| ~ 333
    A = _dev(orc.fill_decay(M, K, tab, 1))
    B = _dev(orc.fill_decay(K, N, tab, 2))
    ctx.normmap_f32(1, B, tile)
    ctx.normmap_f32(0, A, tile)
    tau, ach = ctx.tau_for_ratio(0.05)
    assert tau > 0 and 0.01 < ach < 0.2
    Cref = ctx.multiply(A, B, tile, tau).clone()
    mask, counts, nA, nB = ctx.get_mask(), ctx.get_counts(), ctx.get_normmap(0), ctx.get_normmap(1)
    kept = ctx.get_stats().kept_products
    # the checker's kept set says which A tiles are needed at all: some are not (which matters to a
    # pass that knows it), and some tiles of either operand must be exactly zero
    needed = np.unpackbits(mask.view(np.uint8), axis=-1, bitorder="little")[..., :K // tile].any(axis=1)
    assert 0 < needed.sum() < needed.size
    assert 0 < np.count_nonzero(nB == 0) < nB.size and 0 < np.count_nonzero(nA == 0) < nA.size
    loud = ctx.multiply(torch.full_like(A, 1000.0), torch.full_like(B, 1000.0), tile, 0.0)   # both workspace copies are now loud
    assert float(loud.min()) > 0
    C = ctx.multiply(A, B, tile, tau, prune=True)
    assert torch.equal(C, Cref)
    assert np.array_equal(ctx.get_mask(), mask) and np.array_equal(ctx.get_counts(), counts)
    assert np.array_equal(ctx.get_normmap(0).view(np.uint32), nA.view(np.uint32))
    assert np.array_equal(ctx.get_normmap(1).view(np.uint32), nB.view(np.uint32))
    assert ctx.get_stats().kept_products == kept
    # the incomplete copies are fenced off
    for call in (lambda: ctx.get_fp16(0), lambda: ctx.get_fp16(1), lambda: ctx.error_vs_dense(C),
                 lambda: ctx.multiply(A, B, tile, tau * 0.5, reuse_a=True, reuse_b=True),
                 lambda: ctx.multiply(A, B, tile, tau, reuse_a=True),
                 lambda: ctx.multiply(A, B, tile, 0.0, reuse_b=True)):
        with pytest.raises(sp.SpammError) as ei:
            call()
        assert ei.value.code == -4
    # ... but serve the same operands at the same or a larger threshold
    ctx.multiply(A, B, tile, tau, prune=True)
    C2 = ctx.multiply(A, B, tile, tau * 2, reuse_a=True, reuse_b=True).clone()
    C3 = ctx.multiply(A, B, tile, tau * 0.5, reuse_b=True).clone()        # B's copy serves any tau > 0
    assert torch.equal(C2, ctx.multiply(A, B, tile, tau * 2))
    assert torch.equal(C3, ctx.multiply(A, B, tile, tau * 0.5))
    # and a plain call makes them whole again
    assert np.array_equal(ctx.get_fp16(0), orc.f32_to_f16_bits(A.cpu().numpy()))
    assert np.array_equal(ctx.get_fp16(1), orc.f32_to_f16_bits(B.cpu().numpy()))
    # tau = 0 (nothing may be left out) and tau = inf through the flag
    assert torch.equal(ctx.multiply(A, B, tile, 0.0, prune=True), ctx.multiply(A, B, tile, 0.0))
    assert np.array_equal(ctx.get_fp16(1), orc.f32_to_f16_bits(B.cpu().numpy()))
    assert float(ctx.multiply(A, B, tile, float("inf"), prune=True).abs().max()) == 0.0


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("tile", [32, 64, 128])
@pytest.mark.parametrize("route", ["pair", "b_alone", "a_eq_b"])
def test_passes_without_row_maxima_leave_out_tiles_of_norm_zero_only(orc, ctx, route, tile, half):
    """A tau-aware copy of B (and A's where both are made without row maxima) may lack the tiles of norm zero and no
    others, however large the call's own tau: it serves every tau > 0 afterwards.  The copies are loud before, so
    that a tile that was left out shows in the product that reuses it."""
    import torch
    n = 768
    tab = orc.decay_table("exp", n, 0.05)                     # exactly zero in fp16 beyond |i - j| ~ 333
    A, B = _dev(orc.fill_decay(n, n, tab, 1)), _dev(orc.fill_decay(n, n, tab, 2))
    if half:
        A, B = A.half(), B.half()
    if route == "a_eq_b":
        B = A
    loud = torch.full_like(A, 1000.0)

    def pruned(A, B, tau):
        ctx.multiply(loud, loud, tile, 0.0)
        if route == "b_alone":                                # A resident and whole: B's pass runs by itself
            (ctx.normmap_f16 if half else ctx.normmap_f32)(0, A, tile)
        return ctx.multiply(A, B, tile, tau, prune=True, a_eq_b=route == "a_eq_b", reuse_a=route == "b_alone")

    want = ctx.multiply(A, B, tile, 1e-3).clone()
    assert 0 < np.count_nonzero(ctx.get_normmap(1) == 0) < (n // tile) ** 2
    for tau in (float("inf"), 1e35):
        assert float(pruned(A, B, tau).abs().max()) == 0.0
        one_pass = route == "a_eq_b" and tile != 128          # (its copy of A is B's equal; the pair's serves no smaller tau)
        got = ctx.multiply(A, B, tile, 1e-3, reuse_a=route == "b_alone" or one_pass, reuse_b=True)
        assert torch.equal(got, want), tau
    # an infinite norm keeps every partner of positive norm, also at tau = inf and in the call itself
    A = A.clone()
    A[5, 70] = float("inf")
    if route == "a_eq_b":
        B = A
    want = ctx.multiply(A, B, tile, float("inf")).clone()
    kept = ctx.get_stats().kept_products
    assert 0 < kept < (n // tile) ** 3
    got = pruned(A, B, float("inf"))
    assert ctx.get_stats().kept_products == kept
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("tile", [32, 64, 128])
def test_tau_aware_a_pass_by_row_maxima_gives_the_same_product(orc, ctx, tile, half):
    """A's pass of its own knows B's norms and leaves out every tile that no product keeps (k_rowmax and the bounded
    test): against a resident B, and in a call of more strips than the paired passes take (4096), where B's pass of
    its own runs before it.  Both copies are loud before."""
    import torch
    M, K, N = 1024, 768, 512 + tile
    tab = orc.decay_table("exp", 1024, 0.05)
    A, B = _dev(orc.fill_decay(M, K, tab, 1)), _dev(orc.fill_decay(K, N, tab, 2))
    # the long one: rows of the first, at scales of their own, over 2045 tile rows
    scale = torch.exp2(torch.randint(-6, 1, (2045, 1), generator=torch.Generator().manual_seed(3)).float()).cuda()
    long = (A[:tile].repeat(2045, 1).view(2045, -1) * scale).view(2045 * tile, K)
    for X, resident in ((A, True), (long, False)):
        Y = B
        if half:
            X, Y = X.half(), B.half()
        normmap = ctx.normmap_f16 if half else ctx.normmap_f32
        normmap(1, Y, tile)
        normmap(0, X, tile)
        nA, nB = ctx.get_normmap(0), ctx.get_normmap(1)
        tau = ctx.tau_for_ratio(0.05)[0]
        skipped = np.count_nonzero(nA * nB.max(axis=1)[None, :] < np.float32(tau))
        assert np.count_nonzero(nA == 0) < skipped < nA.size
        want = ctx.multiply(X, Y, tile, tau).clone()
        mask, counts, kept = ctx.get_mask(), ctx.get_counts(), ctx.get_stats().kept_products
        ctx.multiply(torch.full_like(X, 1000.0), torch.full_like(Y, 1000.0), tile, 0.0)
        if resident:
            normmap(1, Y, tile)
        got = ctx.multiply(X, Y, tile, tau, prune=True, reuse_b=resident)
        assert torch.equal(got, want)
        assert np.array_equal(ctx.get_mask(), mask) and np.array_equal(ctx.get_counts(), counts)
        assert ctx.get_stats().kept_products == kept > 0
        assert np.array_equal(ctx.get_normmap(0).view(np.uint32), nA.view(np.uint32))
        want = ctx.multiply(X, Y, tile, tau * 2).clone()
        ctx.multiply(torch.full_like(X, 1000.0), torch.full_like(Y, 1000.0), tile, 0.0)
        ctx.multiply(X, Y, tile, tau, prune=True)
        assert torch.equal(ctx.multiply(X, Y, tile, tau * 2, reuse_a=True, reuse_b=True), want)


def test_fp16_passes_of_three_to_four_strips_per_cu(orc, ctx):
    # fp16 at tile 64, 769 to 1024 strips of 256 columns: strips of 512 in two phases, here ragged (7 1/8 of them), for
    # either role and for both at once, against the paired passes (strips of 256) of the same operands
    import torch
    n, tile = 57 * 64, 64
    tab = orc.decay_table("exp", n, 0.01)
    X = torch.empty((n, n), dtype=torch.float32, device="cuda")
    ctx.fill_decay(X, tab, 1)
    X = X.half()
    bits = X.cpu().numpy().view(np.uint16)
    ctx.multiply(X, X, tile, 1.0)                             # the paired passes
    nA, nB = ctx.get_normmap(0), ctx.get_normmap(1)
    tau = ctx.tau_for_ratio(0.1)[0]
    want = ctx.multiply(X, X, tile, tau).clone()
    ctx.multiply(torch.full_like(X, 1000.0), torch.full_like(X, 1000.0), tile, 0.0)
    for both in (False, True):
        if both:
            got = ctx.multiply(X, X, tile, tau, a_eq_b=True)
        else:
            ctx.normmap_f16(1, X, tile)
            ctx.normmap_f16(0, X, tile)
            ctx.gate(tau)
            got = ctx.gemm_gated(torch.empty_like(want))
        assert np.array_equal(ctx.get_fp16(0), bits) and np.array_equal(ctx.get_fp16(1), bits)
        assert np.array_equal(ctx.get_normmap(0).view(np.uint32), nA.view(np.uint32))
        assert np.array_equal(ctx.get_normmap(1).view(np.uint32), nB.view(np.uint32))
        assert torch.equal(got, want)


@pytest.mark.parametrize("tile", [32, 64, 128])
@pytest.mark.parametrize("half", [False, True])
def test_conversion_on_either_side_of_what_the_caches_keep(ctx, tile, half):
    """Input of more than 32 MiB is read past the caches, less through them, by launches of their own, and strips of nothing but
    zeros are stored past them: a matrix just beyond that line and each of its halves, in both roles, with zero strips, zeros beside
    the smallest value there is and single values; values against the input's, the halves' norms against the whole's, bit for
    bit.  A = B by one read on either side of the line."""
    import torch

    def with_zeros(X):
        X[:tile, 512:1024] = 0.0
        X[tile:2 * tile, :512] = 0.0
        X[tile + 5, 131] = 1.0
        X[-tile:, 1024:1536] = 0.0
        X[-1, 1535] = 2.0 ** -24
        X[:, 2048:2112] = 0.0
        return X.half() if half else X
    rows, cols = 512, (33280 if half else 16640) if tile < 128 else (33024 if half else 16640)
    g = torch.Generator(device="cuda")
    g.manual_seed(tile)
    X = with_zeros(torch.rand((rows, cols), generator=g, device="cuda") * 2.0 - 1.0)
    assert X.numel() * X.element_size() > 32 << 20
    convert = ctx.normmap_f16 if half else ctx.normmap_f32
    bits = X.half().cpu().numpy().view(np.uint16)
    for role in (1, 0):
        whole = None
        for first, last in ((0, rows), (0, rows // 2), (rows // 2, rows)):
            part = X[first:last]
            other = torch.zeros((tile, last - first) if role == 1 else (cols, tile), dtype=X.dtype, device="cuda")
            convert(1 - role, other, tile)
            convert(role, part, tile)
            assert np.array_equal(ctx.get_fp16(role), bits[first:last])
            nm = ctx.get_normmap(role)
            whole = nm if whole is None else whole
            assert np.array_equal(nm.view(np.uint32), whole[first // tile:last // tile].view(np.uint32))
            assert nm.min() == 0.0 < nm.max()
    for n in (2048, 4224 if half else 2944):
        Y = with_zeros(torch.rand((n, n), generator=g, device="cuda") * 2.0 - 1.0)
        two = ctx.multiply(Y, Y.clone(), tile, 0.0)
        maps = ctx.get_normmap(0), ctx.get_normmap(1)
        assert torch.equal(ctx.multiply(Y, Y, tile, 0.0, a_eq_b=True), two)
        for role in (0, 1):
            assert np.array_equal(ctx.get_fp16(role), Y.half().cpu().numpy().view(np.uint16))
            assert np.array_equal(ctx.get_normmap(role).view(np.uint32), maps[role].view(np.uint32))


@pytest.mark.parametrize("rows,N,row0", [(2048, 1024, 64), (512, 512, 0), (4096, 2048, 0), (2112, 960, 0)])
def test_error_report_by_any_block_shape(ctx, rows, N, row0):
    """A wave of the exact product owns 64 x 32 of C (the first case, on 256 CUs), 32 x 32, 64 x 64, or what the grid
    makes best: against a product in fp64 on the host.  Norms of sums of squares in another order: K + rows * N terms
    of 2^-53 each, below 1e-9; the difference's norm is as large as C's (half of the products are dropped)."""
    import torch
    K, tile = 320, 64
    M = row0 + rows
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + N)
    A = torch.rand((M, K), generator=g, device="cuda") * torch.exp2(-torch.arange(K, device="cuda") / 40.0) - 0.3
    B = torch.rand((K, N), generator=g, device="cuda") - 0.5
    ctx.normmap_f32(1, B, tile)
    ctx.normmap_f32(0, A, tile)
    C = ctx.multiply(A, B, tile, ctx.tau_for_ratio(0.5)[0])
    dense = A.half().double().cpu().numpy()[row0:] @ B.half().double().cpu().numpy()
    c = C.cpu().numpy().astype(np.float64)[row0:]
    want = [np.linalg.norm(c - dense), np.linalg.norm(dense), np.linalg.norm(c)]
    assert want[0] > 0.01 * want[1]
    for got, ref in zip(ctx.error_vs_dense(C, row0, M), want):
        assert abs(got - ref) <= 1e-9 * ref


@pytest.mark.parametrize("tile,M,K,N,row0,rows,kind", [
    (32, 64, 32, 64, 0, 64, "unit"), (32, 192, 416, 320, 64, 128, "unit"), (64, 576, 1088, 640, 0, 576, "limbs"),
    (32, 1024, 608, 2304, 128, 832, "limbs"), (128, 4096, 256, 2176, 0, 4096, "limbs"), (64, 512, 32704, 512, 0, 512, "edge"),
    (64, 256, 32768, 256, 0, 256, "edge"), (64, 2048, 320, 1024, 0, 2048, "large"), (128, 512, 512, 512, 0, 512, "large"),
    (64, 8256, 2048, 128, 64, 8192, "limbs"), (64, 576, 1024, 14592, 0, 576, "unit"),        # blocks of C one or few across, or high
    (64, 320, 192, 320, 0, 320, "inf"), (32, 256, 256, 256, 0, 256, "zero"),
    (64, 1280, 1024, 1088, 0, 1280, "inf"), (32, 1184, 1056, 1280, 64, 1088, "nan"), (128, 1280, 1024, 1280, 0, 1280, "zero"),
    (32, 1344, 1056, 1280, 64, 1280, "unit"), (64, 1280, 1024, 1088, 0, 1280, "large"),
    (128, 2048, 512, 2048, 0, 2048, "large"), (32, 2048, 544, 2112, 64, 1984, "inf")])
def test_error_report_over_the_range_of_fp16(ctx, tile, M, K, N, row0, rows, kind):
    """Whatever the magnitudes: 0 to 4 bytes a value by blocks, just inside and outside of what bytes hold, subnormals,
    infinities and NaN, the largest sums that 11 bits a value make at the longest K.  Against fp64 on the host (K terms a sum,
    rows * N in a norm, 2^-53 each, below 1e-9); the exact product of whole multiples of 2^-24 is what both sides form.
    Whole numbers from K = 256 on where the split is worth it, and one shape or two of every kind on the other side of that."""
    import torch
    rng = np.random.default_rng(M + K + N)

    def operand(r, c):
        X = rng.uniform(-1.0, 1.0, (r, c))
        if kind == "limbs":       # 64 x 64 blocks of every magnitude that needs 0 to 4 bytes, and what lies below fp16
            X *= np.kron(np.exp2(rng.choice([-40, -22, -16, -15, -9, -8, -1, 0, 6], (-(-r // 64), -(-c // 64)))), np.ones((64, 64)))[:r, :c]
        elif kind == "edge":      # digits (0, 0, -128, 127) and (0, -128, -127, 1), of one sign: an order's sum reaches 8e8, 0.37 of 2^31
            X = np.where(X < 0, -126.5, 126.5)
            X[:, ::2] = np.where(X[:, ::2] < 0, -0.50196, 0.50196)
        elif kind == "large":
            X *= 60000.0
        return X.astype(np.float32)

    A, B = operand(M, K), operand(K, N)
    if kind == "edge":
        A, B = np.abs(A), np.abs(B)
    if kind == "zero":
        A[:] = 0
    if kind in ("inf", "nan"):
        A[70, 100] = np.inf if kind == "inf" else np.nan
    hA, hB = A.astype(np.float16).astype(np.float64), B.astype(np.float16).astype(np.float64)
    ctx.normmap_f32(1, torch.from_numpy(B).cuda(), tile)
    ctx.normmap_f32(0, torch.from_numpy(A).cuda(), tile)
    with np.errstate(invalid="ignore"):
        dense = hA[row0:row0 + rows] @ hB
    C = np.zeros((M, N), dtype=np.float32)
    C[row0:row0 + rows] = (0.75 * np.nan_to_num(dense, nan=1.0, posinf=1.0, neginf=1.0)).astype(np.float32)
    c = C[row0:row0 + rows].astype(np.float64)
    for _ in range(2):            # (the second call finds the workspace as the first left it)
        got = ctx.error_vs_dense(torch.from_numpy(C).cuda(), row0, row0 + rows)
        if kind in ("inf", "nan"):
            assert not np.isfinite(got[0]) and not np.isfinite(got[1])
            assert abs(got[2] - np.linalg.norm(c)) <= 1e-9 * np.linalg.norm(c)
            continue
        for g, ref in zip(got, (np.linalg.norm(c - dense), np.linalg.norm(dense), np.linalg.norm(c))):
            assert abs(g - ref) <= 1e-9 * ref


@pytest.mark.parametrize("K", [4096 - 32, 4096, 64 * 66, 16384 + 64])
def test_error_report_by_steps_of_every_kind(ctx, K):
    """Blocks of 64 k that need 0 to 4 bytes on either side, drawn so that every pair of them occurs an odd number of times here and
    an even one there: steps with one block, some and all they can hold, 64 steps and more of one block of C, a last
    block of 32 k.  The exact product of whole multiples of 2^-24 on both sides; sums of squares in another order, 1e-9."""
    import torch
    rng = np.random.default_rng(K)
    M = N = 512
    nkb = -(-K // 64)

    def scales(n):
        s = np.exp2(rng.choice([-40.0, -20.0, -12.0, -4.0, 5.0], (8, n), p=[0.1, 0.25, 0.25, 0.25, 0.15]))
        return np.kron(s, np.ones((64, 64)))[:, :K]
    A = (rng.uniform(-1.0, 1.0, (M, K)) * scales(nkb)).astype(np.float16)
    B = (rng.uniform(-1.0, 1.0, (K, N)) * scales(nkb).T).astype(np.float16)
    dense = A.astype(np.float64) @ B.astype(np.float64)
    C = (0.75 * dense).astype(np.float32)
    ctx.normmap_f16(1, torch.from_numpy(B).cuda(), 32)
    ctx.normmap_f16(0, torch.from_numpy(A).cuda(), 32)
    got = ctx.error_vs_dense(torch.from_numpy(C).cuda())
    for g, ref in zip(got, (np.linalg.norm(C - dense), np.linalg.norm(dense), np.linalg.norm(C.astype(np.float64)))):
        assert abs(g - ref) <= 1e-9 * ref


def test_error_report_rounds_once(ctx):
    """21800 products of 257 / 512 with itself, 10900 of minus twice that by values with other digits, and one of 2^-24 with
    itself: the upper and the lower orders of a sum pass 2^53 and cancel, and what is left is the last product."""
    import torch
    K = 32704
    a, b = np.zeros(K), np.zeros(K)
    a[:21800] = b[:21800] = 257 / 512
    a[21800:32700], b[21800:32700] = -64.25, 257 * 2.0 ** -15
    a[32700] = b[32700] = 2.0 ** -24
    ctx.normmap_f16(1, torch.from_numpy(np.repeat(b[:, None], 64, axis=1).astype(np.float16)).cuda(), 32)
    ctx.normmap_f16(0, torch.from_numpy(np.repeat(a[None], 64, axis=0).astype(np.float16)).cuda(), 32)
    C = torch.full((64, 64), 2.0 ** -48, dtype=torch.float32, device="cuda")
    assert ctx.error_vs_dense(C) == (0.0, 64 * 2.0 ** -48, 64 * 2.0 ** -48)


@pytest.mark.parametrize("M,K,N,tile", [(1280, 1024, 1088, 64), (2048, 512, 2048, 128)])
def test_error_reports_of_small_and_large_values_by_turns(ctx, M, K, N, tile):
    """Values that are too large are taken by the integer product's launch, or by another when it has said so: report after
    report, of one kind and the other, each on another stream than the last and none waited for."""
    import torch
    rng = np.random.default_rng(5)
    A, B = rng.uniform(-1.0, 1.0, (M, K)).astype(np.float16), rng.uniform(-1.0, 1.0, (K, N)).astype(np.float16)
    C = rng.uniform(-1.0, 1.0, (M, N)).astype(np.float32)
    dB, dC = torch.from_numpy(B).cuda(), torch.from_numpy(C).cuda()
    kinds = []
    for scale in (1, 1024):                       # (a power of two: fp16 holds the scaled values too)
        X = A * np.float16(scale)
        dense = X.astype(np.float64) @ B.astype(np.float64)
        kinds.append((torch.from_numpy(X).cuda(), [np.linalg.norm(v) for v in (C - dense, dense, C.astype(np.float64))]))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for at, kind in enumerate((0, 1, 0, 0, 1, 1, 0, 1)):
        ctx.set_stream(streams[at % 2].cuda_stream)
        ctx.normmap_f16(1, dB, tile)
        ctx.normmap_f16(0, kinds[kind][0], tile)
        for got, want in zip(ctx.error_vs_dense(dC), kinds[kind][1]):
            assert abs(got - want) <= 1e-9 * want, at
    torch.cuda.synchronize()
    ctx.set_stream(None)


def test_native_multiply_call_answers_as_the_checks_in_python(ctx):
    """The multiply calls take usual arguments through native code and leave all others to the checks in Python: with and without it the
    same results and the same errors, and nothing of a refused call remains."""
    import types
    import torch
    from cuspamm_amd import api
    N, tile = 256, 32
    g = torch.Generator(device="cuda").manual_seed(5)
    A = torch.randn((N, N), generator=g, device="cuda")
    B = torch.randn((N, 2 * N), generator=g, device="cuda")
    h = A.half()
    C = torch.empty((N, 2 * N), device="cuda")
    none = types.SimpleNamespace(multiply=lambda *a: None, multiply_noalloc=lambda *a: None)
    calls = [lambda: ctx.multiply(A, B, tile, 4.0, C), lambda: ctx.multiply(A, B, tile, 4.0, C=C, prune=True), lambda: ctx.multiply(A, B, tile, 4),
             lambda: ctx.multiply(A, B, np.int64(tile), np.float32(4.0), C), lambda: ctx.multiply(h, B.half(), tile, 4.0, C),
             lambda: ctx.multiply(A, B, tile, 4.0, C, reuse_b=True), lambda: ctx.multiply(A, A, tile, 4.0, a_eq_b=True),
             lambda: ctx.multiply_noalloc(A, B, tile, 4.0, C), lambda: ctx.multiply_noalloc(A, B, tile, 4.0, C, timing=True),
             lambda: ctx.multiply(A.requires_grad_(False), torch.nn.Parameter(B), tile, 4.0, C),
             # refused: by the checks, or by the engine
             lambda: ctx.multiply(A, B.t(), tile, 4.0, C), lambda: ctx.multiply(A.t(), B, tile, 4.0, C), lambda: ctx.multiply(A, B, tile, 4.0, C[:, :N]),
             lambda: ctx.multiply(A, B, tile, 4.0, C.cpu()), lambda: ctx.multiply(A.cpu(), B, tile, 4.0, C), lambda: ctx.multiply(A, B.half(), tile, 4.0, C),
             lambda: ctx.multiply(A.double(), B.double(), tile, 4.0, C), lambda: ctx.multiply(A, B, tile, 4.0, C.half()), lambda: ctx.multiply(A[0], B, tile, 4.0, C),
             lambda: ctx.multiply(A, B, 48, 4.0, C), lambda: ctx.multiply(A, B, 0, 4.0, C), lambda: ctx.multiply(A, B, "32", "x", C),
             lambda: ctx.multiply(A, B, tile, float("nan"), C), lambda: ctx.multiply(A, B, tile, None, C), lambda: ctx.multiply(A, B, tile, 4.0, "C"),
             lambda: ctx.multiply(A, B, tile, 4.0, C, a_eq_b=True), lambda: ctx.multiply_noalloc(h, B.half(), tile, 4.0, C),
             lambda: ctx.multiply_noalloc(A, B, tile, 4.0, None)]

    def outcome(call):
        ctx.multiply(A, B, tile, 4.0, C)                          # (what reuse_b refers to)
        C.fill_(float("nan"))
        try:
            out = call().clone()
            return out, ctx._shape, ctx.get_mask()
        except Exception as e:
            return type(e), str(e), ctx._shape

    native, seen = api._call, 0
    for i, call in enumerate(calls):
        first = outcome(call)
        api._call = none
        try:
            second = outcome(call)
        finally:
            api._call = native
        if isinstance(first[0], torch.Tensor):
            seen += 1
            assert torch.equal(first[0], second[0]) and first[1] == second[1] and np.array_equal(first[2], second[2]), i
        else:
            assert first == second, (i, first, second)
    assert seen == 10
    assert native.multiply(None, A, B, C, tile, 4.0, False, False, False, False, False) is None and native.multiply(1, A, B) is None


@pytest.mark.parametrize("lengths", [(256,) * 256, (256,) * 255 + (128,)], ids=["even rows", "ragged rows"])
def test_nested_matrices_are_refused(ctx, lengths):
    """Nested tensors of exactly torch's type, strided, contiguous and two-dimensional: torch throws at their sizes, or answers."""
    import torch
    X = torch.randn((256, 256), device="cuda")
    C = torch.full((256, 256), 7.0, device="cuda")
    nested = torch.nested.nested_tensor([X[i, :n] for i, n in enumerate(lengths)])
    assert type(nested) is torch.Tensor and nested.dim() == 2 and nested.is_cuda
    for A, B, out in ((nested, X, C), (X, nested, C), (X, X, nested)):
        for multiply in (ctx.multiply, ctx.multiply_noalloc):
            with pytest.raises((RuntimeError, ValueError)) as e:
                multiply(A, B, 32, 4.0, out)
            assert not hasattr(e.value, "code")                   # (by torch or the checks: the engine was not called)
    assert (C == 7.0).all()
