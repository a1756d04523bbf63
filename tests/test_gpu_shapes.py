"""Shape sweep: ragged tile counts, extreme aspect ratios, long k, special values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
C_REL_TOL = 1e-3


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _check(orc, ctx, A, B, tile, tau):
    import torch
    M, N = A.shape[0], B.shape[1]
    C = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    ctx.multiply(_dev(A), _dev(B), tile, tau, C=C)
    ref = orc.spamm(A, B, tile, tau)
    assert np.array_equal(ctx.get_mask(), ref["mask"])
    assert np.array_equal(ctx.get_counts(), ref["counts"])
    assert ctx.get_stats().kept_products == ref["kept"]
    Cg = C.cpu().numpy()
    err, nrm, _ = orc.frob_diff(Cg, ref["C"])
    assert err <= C_REL_TOL * nrm or (nrm == 0 and err == 0)
    return ref


@pytest.mark.usefixtures("work_unit")
def test_random_shapes(orc, ctx):
    rng = np.random.default_rng(2024)
    for trial in range(40):
        tile = int(rng.choice([32, 64, 128]))
        M, K, N = (int(rng.integers(1, 1 + 1024 // tile)) * tile for _ in range(3))
        lam = float(rng.choice([0.0, 0.005, 0.02, 0.1]))
        tab = orc.decay_table("exp", max(M, K, N), lam)
        A = orc.fill_decay(M, K, tab, 10 + trial)
        B = orc.fill_decay(K, N, tab, 100 + trial)
        nA = orc.normmap(orc.f32_to_f16_bits(A), tile, 0)
        nB = orc.normmap(orc.f32_to_f16_bits(B), tile, 1)
        ratio = float(rng.choice([0.0, 0.1, 0.5, 0.9, 1.0]))
        tau = 0.0 if ratio == 1.0 else (np.inf if ratio == 0.0 else orc.tau_for_ratio(nA, nB, ratio)[0])
        _check(orc, ctx, A, B, tile, tau)


@pytest.mark.parametrize("M,K,N,tile", [(64, 64, 8192, 64), (8192, 64, 64, 64), (64, 16384, 64, 32),
                                        (128, 32768, 128, 128), (2560, 256, 2304, 64), (32, 32, 32, 32),
                                        (288, 32, 2080, 32),
                                        (64, 576, 102400, 64),     # the reference's im2col shape (para.h:20-21)
                                        (32, 288000, 32, 32),      # 9000 k tiles: bitmaps beyond 64 KiB of LDS
                                        (64, 65535 * 64, 64, 64),  # the most k tiles the ABI takes
                                        (32, 65535 * 32, 32, 32)])  # ... at tile 32: the gate walks k in four chunks
def test_extreme_aspect_ratios(orc, ctx, work_unit, M, K, N, tile):
    tab = orc.decay_table("exp", max(M, K, N), 0.002)
    A = orc.fill_decay(M, K, tab, 1)
    B = orc.fill_decay(K, N, tab, 2)
    nA = orc.normmap(orc.f32_to_f16_bits(A), tile, 0)
    nB = orc.normmap(orc.f32_to_f16_bits(B), tile, 1)
    tau, _ = orc.tau_for_ratio(nA, nB, 0.4)
    ref = _check(orc, ctx, A, B, tile, tau)
    assert 0 < ref["kept"]


@pytest.mark.parametrize("M,n_sup_n,percents", [(256, 520, (100, 40, 10)), (1088, 1030, (100, 30))])
def test_more_than_512_super_tiles_of_c(orc, ctx, M, n_sup_n, percents):
    # beyond 512 super tiles the schedule ranks them by sorting indices padded to a power of two:
    # 1 x 520 -> 1024, and 2 x 1030 = 2060 -> 4096 (M = 1088 is five macro tile rows, the fifth
    # starts a second row of super tiles; 9 GB of C).  B's non-zero column range is cut so that all,
    # 40 % and 10 % of the 520 super tiles hold work -- one case per way of dealing; beyond 2048
    # super tiles there is one way only
    K, tile = 64, 64
    N = n_sup_n * 8 * 256
    tab = orc.decay_table("exp", N, 0.0)
    A = orc.fill_decay(M, K, tab, 1)
    B = orc.fill_decay(K, N, tab, 2)
    for percent in percents:
        cut = N * percent // 100          # a multiple of the tile size
        B[:, cut:] = 0.0
        ref = _check(orc, ctx, A, B, tile, 1e-30)
        assert ref["kept"] == (M // tile) * (cut // tile)


@pytest.mark.parametrize("chunk_words", [1, 3])
def test_gate_in_small_k_chunks_gives_the_same_lists(orc, ctx, chunk_words):
    """A macro tile's bitmaps normally fit a CU's LDS whole; beyond ~19 500 k tiles (tile 32) the
    gate walks k in chunks, twice.  Forcing chunks of 1 and 3 words (64 and 192 k tiles) sends
    ordinary shapes down that path: mask, counts, kept total and C must not change by a bit."""
    import torch
    import cuspamm_amd as sp
    other = sp.SpammContext(0)
    other.set_option(sp.OPT_GATE_CHUNK_WORDS, chunk_words)
    try:
        for (M, K, N), tile, lam, ratio in [((512, 8192, 768), 32, 0.004, 0.3), ((1024, 12800, 512), 64, 0.001, 0.5),
                                            ((256, 33280, 384), 128, 0.0005, 0.4), ((320, 6432, 288), 32, 0.0, 1.0)]:
            tab = orc.decay_table("exp", max(M, K, N), lam)
            dA = torch.empty((M, K), dtype=torch.float32, device="cuda")
            dB = torch.empty((K, N), dtype=torch.float32, device="cuda")
            ctx.fill_decay(dA, tab, 1)
            ctx.fill_decay(dB, tab, 2)
            ctx.normmap_f32(1, dB, tile)
            ctx.normmap_f32(0, dA, tile)
            tau = 0.0 if ratio == 1.0 else ctx.tau_for_ratio(ratio)[0]
            want = ctx.multiply(dA, dB, tile, tau)
            mask, counts, kept = ctx.get_mask(), ctx.get_counts(), ctx.get_stats().kept_products
            got = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
            other.multiply(dA, dB, tile, tau, C=got)
            assert np.array_equal(other.get_mask(), mask)
            assert np.array_equal(other.get_counts(), counts)
            assert other.get_stats().kept_products == kept and 0 < kept
            assert torch.equal(got, want)
        tab = orc.decay_table("exp", 2048, 0.003)
        _check(orc, other, orc.fill_decay(384, 2048, tab, 3), orc.fill_decay(2048, 320, tab, 4), 32, 0.05)
    finally:
        other.close()


@pytest.mark.parametrize("tile,nbM,nbK,nbN", [(32, 8, 64, 8), (32, 9, 65, 23), (32, 16, 257, 8), (32, 3, 4161, 5), (64, 4, 1, 4), (64, 7, 128, 9),
                                              (64, 8, 513, 4), (64, 5, 8200, 3), (128, 2, 63, 2), (128, 5, 256, 3), (128, 3, 321, 7)])
def test_gate_by_bits_of_a_lane_gives_the_same_lists(ctx, tile, nbM, nbK, nbN):
    """The gate of a macro tile whose bitmaps fit LDS against the one that walks k in chunks, and against numpy: words
    held in registers and in LDS, one word to more than a wave's lanes, the last one cut, macro tiles cut by the matrix, norms
    that are zero, infinite, negative or NaN, products that overflow or are denormal, every kind of tau.  Where operands
    are small enough, C, whose bits depend on the lists, as well."""
    import torch
    import cuspamm_amd as sp
    rng = np.random.default_rng(nbK)
    nA = rng.random((nbM, nbK), dtype=np.float32) * np.exp(-0.02 * rng.integers(0, 400, (1, nbK))).astype(np.float32)
    nB = rng.random((nbK, nbN), dtype=np.float32)
    nA[:, : nbK // 2 // 64 * 64] *= np.float32(1e-30)                 # words with nothing kept, at most of the taus
    other = sp.SpammContext(0)
    other.set_option(sp.OPT_GATE_CHUNK_WORDS, 3)
    plain = sp.SpammContext(0)
    plain.set_option(sp.OPT_GEMM_SHAPE, 1)
    try:
        for special in (False, True):
            if special:
                odd = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, -1.0, 3e38, 1e-40], np.float32)
                for X in (nA, nB):
                    at = rng.random(X.shape) < 0.02
                    X[at] = rng.choice(odd, at.sum())
            at_tau = float(nA[0, -1] * nB[-1, 0])
            for tau in (0.0, 0.3, 1e-33, 0.1 if at_tau != at_tau else at_tau, -1.0, float("inf")):
                got = []
                for c in (plain, other):
                    c.set_normmaps(nA, nB, tile)
                    c.gate(tau)
                    got.append((c.get_mask(), c.get_counts(), c.get_macro_counts()[0], c.get_stats().kept_products))
                with np.errstate(all="ignore"):
                    keep = nA[:, None, :] * nB.T[None, :, :] >= np.float32(tau)
                assert np.array_equal(got[0][1], keep.sum(axis=2)) and got[0][3] == keep.sum()
                for x, y in zip(*got):
                    assert np.array_equal(x, y)
        if nbK <= 600:
            M, K, N = nbM * tile, nbK * tile, nbN * tile
            A = torch.randn((M, K), device="cuda") * (torch.rand((nbM, 1, nbK, 1), device="cuda") < 0.6).expand(-1, tile, -1, tile).reshape(M, K)
            B = torch.randn((K, N), device="cuda") * torch.logspace(0, -4, nbN, device="cuda").repeat_interleave(tile)
            for tau in (0.0, 0.05 * tile, 1.02 * tile):
                assert torch.equal(plain.multiply(A, B, tile, tau), other.multiply(A, B, tile, tau))
    finally:
        plain.close()
        other.close()


@pytest.mark.parametrize("shape", [2, 3, 4])
def test_other_gemm_work_units_give_the_same_product(orc, ctx, shape):
    """The GEMM's work unit is a whole 256 x 256 macro tile by four waves (shape 1), a 128 x 256
    half by four waves, two workgroups per CU (2), a whole macro tile by eight waves (3), or shape 1
    by workgroups that stay and draw macro tiles from a ticket counter per XCD (4; every case runs
    twice on one gate, so the counter must be back at zero after a launch).  All
    walk the macro tile's list in the same order, so C must agree bit for bit -- whole macro tiles,
    ragged edges where the lower half lies beyond the matrix, all three tile sizes, dense and empty
    regions -- and with the checker."""
    import torch
    import cuspamm_amd as sp
    other = sp.SpammContext(0)
    other.set_option(sp.OPT_GEMM_SHAPE, shape)
    ctx.set_option(sp.OPT_GEMM_SHAPE, 1)
    try:
        for (M, K, N), tile, lam, ratio in [((2304, 1024, 4352), 64, 0.004, 0.3), ((1280, 512, 768), 32, 0.01, 0.5),
                                            ((2048, 2048, 2048), 128, 0.002, 0.2), ((1024, 256, 1280), 64, 0.0, 1.0),
                                            ((384, 2048, 320), 32, 0.003, 0.4), ((128, 1024, 128), 128, 0.0, 1.0),
                                            ((640, 4096, 896), 128, 0.001, 0.1), ((4096, 4096, 4096), 64, 0.01, 0.05),
                                            ((96, 64, 160), 32, 0.0, 1.0)]:
            tab = orc.decay_table("exp", max(M, K, N), lam)
            dA = torch.empty((M, K), dtype=torch.float32, device="cuda")
            dB = torch.empty((K, N), dtype=torch.float32, device="cuda")
            ctx.fill_decay(dA, tab, 1)
            ctx.fill_decay(dB, tab, 2)
            ctx.normmap_f32(1, dB, tile)
            ctx.normmap_f32(0, dA, tile)
            tau = 0.0 if ratio == 1.0 else ctx.tau_for_ratio(ratio)[0]
            want = ctx.multiply(dA, dB, tile, tau)
            mask, kept = ctx.get_mask(), ctx.get_stats().kept_products
            got = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
            other.multiply(dA, dB, tile, tau, C=got)
            assert np.array_equal(other.get_mask(), mask)
            assert other.get_stats().kept_products == kept and 0 < kept
            assert torch.equal(got, want), (M, K, N, tile)
            got.fill_(float("nan"))
            other.gemm_gated(got)            # the same gate again
            assert torch.equal(got, want), (M, K, N, tile, "second launch on one gate")
        tab = orc.decay_table("exp", 2048, 0.003)
        _check(orc, other, orc.fill_decay(384, 2048, tab, 3), orc.fill_decay(2048, 320, tab, 4), 32, 0.05)
        _check(orc, other, orc.fill_decay(640, 1024, tab, 5), orc.fill_decay(1024, 384, tab, 6), 128, 20.0)
        _check(orc, other, orc.fill_decay(320, 1024, tab, 7), orc.fill_decay(1024, 576, tab, 8), 64, 1.0)
    finally:
        ctx.set_option(sp.OPT_GEMM_SHAPE, 0)
        other.close()


@pytest.mark.usefixtures("work_unit")
def test_scattered_sparsity_pattern(orc, ctx):
    # no band structure at all: random tiles zeroed, so k lists are ragged and macro tiles mixed
    rng = np.random.default_rng(7)
    n, tile = 1024, 64
    A = rng.uniform(-1, 1, size=(n, n)).astype(np.float32)
    B = rng.uniform(-1, 1, size=(n, n)).astype(np.float32)
    za = rng.random((n // tile, n // tile)) < 0.6
    zb = rng.random((n // tile, n // tile)) < 0.6
    A *= np.kron(~za, np.ones((tile, tile), dtype=np.float32))
    B *= np.kron(~zb, np.ones((tile, tile), dtype=np.float32))
    scale = 10.0 ** rng.integers(-3, 1, size=(n // tile, n // tile))
    A *= np.kron(scale, np.ones((tile, tile))).astype(np.float32)
    ref = _check(orc, ctx, A, B, tile, 1.0)
    assert 0 < ref["kept"] < (n // tile) ** 3 // 2


@pytest.mark.usefixtures("work_unit")
def test_non_finite_inputs_follow_ieee_compare(orc, ctx):
    # inf tile norm: kept against any non-zero tile; NaN product (inf*0, NaN norm) is dropped
    n, tile = 256, 64
    rng = np.random.default_rng(3)
    A = rng.uniform(-1, 1, size=(n, n)).astype(np.float32)
    B = rng.uniform(-1, 1, size=(n, n)).astype(np.float32)
    A[5, 70] = 1e6            # overflows fp16 -> inf in tile (0,1)
    A[130, 200] = np.nan      # NaN in tile (2,3)
    B[64:128, 0:64] = 0       # zero tile (1,0): inf * 0 = NaN -> dropped
    import torch
    C = torch.empty((n, n), dtype=torch.float32, device="cuda")
    ctx.multiply(_dev(A), _dev(B), tile, 0.5, C=C)
    ref = orc.spamm(A, B, tile, 0.5)
    assert np.array_equal(ctx.get_mask(), ref["mask"])
    assert np.array_equal(ctx.get_counts(), ref["counts"])
    Cg, Cr = C.cpu().numpy(), ref["C"]
    assert np.array_equal(np.isnan(Cg), np.isnan(Cr))
    assert np.array_equal(np.isinf(Cg), np.isinf(Cr))
    fin = np.isfinite(Cr)
    assert np.linalg.norm(Cg[fin] - Cr[fin]) <= C_REL_TOL * np.linalg.norm(Cr[fin])
    assert not ref["mask"][0, 0, 0] & np.uint64(2)      # (i=0, j=0, k=1): inf * 0 is not kept


@pytest.mark.parametrize("n_xcd", [1, 2, 4])
def test_schedule_for_other_xcd_counts_gives_the_same_product(orc, ctx, work_unit, n_xcd):
    """The GEMM schedule is built for the device's XCD count (8 on a whole MI355X); a partitioned
    device, or one that is not whole XCDs of 32 CUs, gets 4 / 2 / 1 sequences.  The schedule only
    decides where and when a macro tile runs: mask and C must not change by a bit."""
    import torch
    import cuspamm_amd as sp
    other = sp.SpammContext(0)
    other.set_option(sp.OPT_NUM_XCD, n_xcd)
    other.set_option(sp.OPT_GEMM_SHAPE, work_unit)
    try:
        # (the last case is a narrow band over 128 super tiles: the grouped row-major deal)
        for (M, K, N), tile, lam, ratio in [((2304, 1024, 4352), 64, 0.004, 0.3), ((1280, 512, 768), 32, 0.01, 0.5),
                                            ((2048, 2048, 2048), 128, 0.002, 0.2), ((8192, 256, 10240), 64, 0.0, 1.0),
                                            ((16384, 16384, 16384), 64, 0.003, 0.1)]:
            tab = orc.decay_table("exp", max(M, K, N), lam)
            dA = torch.empty((M, K), dtype=torch.float32, device="cuda")
            dB = torch.empty((K, N), dtype=torch.float32, device="cuda")
            ctx.fill_decay(dA, tab, 1)
            ctx.fill_decay(dB, tab, 2)
            ctx.normmap_f32(1, dB, tile)
            ctx.normmap_f32(0, dA, tile)
            tau = 0.0 if ratio == 1.0 else ctx.tau_for_ratio(ratio)[0]
            want = ctx.multiply(dA, dB, tile, tau)
            mask = ctx.get_mask()
            got = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
            other.multiply(dA, dB, tile, tau, C=got)
            assert np.array_equal(other.get_mask(), mask)
            assert torch.equal(got, want)
            del want, got, dA, dB
        tab = orc.decay_table("exp", 1024, 0.01)
        _check(orc, other, orc.fill_decay(768, 1024, tab, 3), orc.fill_decay(1024, 640, tab, 4), 64, 0.3)
    finally:
        other.close()


@pytest.mark.parametrize("M,K,N,tile", [(32, 32, 32, 32), (256, 256, 256, 32), (96, 2080, 224, 32), (416, 160, 736, 32),
                                        (1056, 1568, 1312, 32), (2048, 4096, 1024, 32), (256, 65536, 288, 32),
                                        (64, 64, 64, 64), (320, 8192, 448, 64), (1152, 640, 2112, 64), (1024, 8192, 4096, 64),
                                        (128, 128, 128, 128), (384, 1280, 640, 128), (1920, 512, 2176, 128)])
def test_small_outputs_in_one_launch_give_the_same_product(orc, ctx, M, K, N, tile):
    """Small outputs are gated and multiplied by one kernel, in units of 128 or 64: same mask, counts, kept total
    and, bit for bit, the same C as the gate and the GEMM apart -- units cut by the edges of C, units smaller
    than a tile, one to many 64-k words, empty, sparse, half-full and full lists, both input types."""
    import torch
    import cuspamm_amd as sp
    apart = sp.SpammContext(0)
    apart.set_option(sp.OPT_GEMM_SHAPE, 1)
    try:
        tab = orc.decay_table("exp", max(M, K, N), 12.0 / max(M, K, N))
        dA = torch.empty((M, K), dtype=torch.float32, device="cuda")
        dB = torch.empty((K, N), dtype=torch.float32, device="cuda")
        ctx.fill_decay(dA, tab, 1)
        ctx.fill_decay(dB, tab, 2)
        ctx.normmap_f32(1, dB, tile)
        ctx.normmap_f32(0, dA, tile)
        for tau in (0.0, float("inf"), ctx.tau_for_ratio(0.03)[0], ctx.tau_for_ratio(0.4)[0]):
            for a, b in ((dA, dB), (dA.half(), dB.half())):
                want = apart.multiply(a, b, tile, tau)
                got = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
                ctx.multiply(a, b, tile, tau, C=got)
                assert torch.equal(got, want), tau
                assert np.array_equal(ctx.get_mask(), apart.get_mask()) and np.array_equal(ctx.get_counts(), apart.get_counts())
                assert ctx.get_stats().kept_products == apart.get_stats().kept_products
        # once more on the operands that lie there (no pass runs), then the stages of their own on that gate
        ctx.multiply(dA.half(), dB.half(), tile, tau, C=got, reuse_a=True, reuse_b=True)
        assert torch.equal(got, want) and ctx.get_stats().kept_products == apart.get_stats().kept_products
        assert np.array_equal(ctx.get_macro_counts()[0], apart.get_macro_counts()[0])
        got.fill_(float("nan"))
        assert torch.equal(ctx.gemm_gated(got), want)
    finally:
        apart.close()


@pytest.mark.parametrize("words_k", [31, 32, 33, 63, 64, 65, 127, 128, 129, 256, 257])
@pytest.mark.parametrize("M,N", [(96, 160), (2080, 1952)])
def test_small_outputs_list_every_place_of_a_word(orc, ctx, M, N, words_k):
    """Units of 64 and of 128: a word of 64 k that is the list's only one, or the first or last of several, with its places up to
    the 32nd and the 64th kept, all of them and every other one."""
    test_small_outputs_in_one_launch_give_the_same_product(orc, ctx, M, 32 * words_k, N, 32)


@pytest.mark.parametrize("M,K,N,tile", [(2944, 256, 2912, 32),      # 529 units: no longer two to a CU at once
                                        (3200, 160, 3072, 32), (3200, 256, 3200, 64),               # 600 and 625: two and three to a CU
                                        (3200, 12320, 3136, 32),    # a list too long for three to a CU
                                        (4096, 512, 2560, 64), (4352, 320, 4160, 64),               # dense too: 160 and 289 macro tiles
                                        (4096, 96, 4096, 32), (3968, 384, 4224, 128), (4096, 64, 6144, 64),
                                        (3712, 8192, 3712, 64), (4096, 8192, 4096, 128),            # 841 and 1024 units at their longest
                                        (3712, 8256, 3712, 64), (4096, 12288, 3584, 128),           # beyond it: gate and GEMM
                                        (192, 640, 98304, 64)])     # 1536 units, the most
def test_middling_outputs_in_one_launch_give_the_same_product(orc, ctx, M, K, N, tile):
    test_small_outputs_in_one_launch_give_the_same_product(orc, ctx, M, K, N, tile)


@pytest.mark.parametrize("M,K,N,tile", [(192, 64, 320, 64), (1088, 4032, 832, 64), (1152, 4096, 2112, 64), (2048, 4160, 1088, 64),
                                        (256, 128, 384, 128), (640, 8064, 1152, 128), (1920, 8192, 2176, 128), (1920, 8320, 2176, 128),
                                        (3200, 64, 3264, 64), (3264, 2048, 3136, 64), (3200, 128, 3200, 128),
                                        (3200, 16416, 3136, 32)])   # (a list too long for three units to a CU)
def test_one_word_of_k_tiles_at_its_ends(orc, ctx, M, K, N, tile):
    """The kernel whose list is a register, at one k tile, at 63 and 64 and the other one at 65, by every size of unit and two and
    three units to a CU; stages of its own here (a gate that forms no list), too."""
    import torch
    test_small_outputs_in_one_launch_give_the_same_product(orc, ctx, M, K, N, tile)
    tab = orc.decay_table("exp", max(M, K, N), 12.0 / max(M, K, N))
    dA = torch.empty((M, K), dtype=torch.float32, device="cuda")
    dB = torch.empty((K, N), dtype=torch.float32, device="cuda")
    ctx.fill_decay(dA, tab, 1)
    ctx.fill_decay(dB, tab, 2)
    ctx.normmap_f32(1, dB, tile)
    ctx.normmap_f32(0, dA, tile)
    tau = ctx.tau_for_ratio(0.2)[0]
    want = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    ctx.multiply(dA, dB, tile, tau, C=want)
    mask, counts, kept = ctx.get_mask(), ctx.get_counts(), ctx.get_stats().kept_products
    ctx.gate(float("inf"))
    ctx.gate(tau)
    assert np.array_equal(ctx.get_mask(), mask) and np.array_equal(ctx.get_counts(), counts) and ctx.get_stats().kept_products == kept
    assert torch.equal(ctx.gemm_gated(torch.full_like(want, float("nan"))), want)


@pytest.mark.parametrize("M,K,N,tile", [(3712, 2048, 3712, 32), (3712, 2080, 3712, 32), (4096, 4096, 3584, 64), (4096, 4160, 3584, 64),
                                        (4096, 4096, 4096, 128), (4096, 4224, 4096, 128)])
def test_stages_on_either_side_of_their_line(orc, ctx, M, K, N, tile):
    """Gate, then multiply, by the one-launch kernel's two halves up to one word of 64 k and K = 4096, by the gate and the GEMM
    beyond: mask, counts and, bit for bit, C as by the latter."""
    import torch
    import cuspamm_amd as sp
    apart = sp.SpammContext(0)
    apart.set_option(sp.OPT_GEMM_SHAPE, 1)
    try:
        tab = orc.decay_table("exp", max(M, K, N), 12.0 / max(M, K, N))
        dA = torch.empty((M, K), dtype=torch.float32, device="cuda")
        dB = torch.empty((K, N), dtype=torch.float32, device="cuda")
        ctx.fill_decay(dA, tab, 1)
        ctx.fill_decay(dB, tab, 2)
        for c in (ctx, apart):
            c.normmap_f32(1, dB, tile)
            c.normmap_f32(0, dA, tile)
        for tau in (ctx.tau_for_ratio(0.03)[0], ctx.tau_for_ratio(0.4)[0], float("inf")):
            out = []
            for c in (ctx, apart):
                C = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
                c.gate(tau)
                before = c.get_mask(), c.get_counts()
                out.append((c.gemm_gated(C), before, c.get_stats().kept_products))
            (C, maps, kept), (C2, maps2, kept2) = out
            assert torch.equal(C, C2) and kept == kept2
            assert all(np.array_equal(x, y) for x, y in zip(maps, maps2))
    finally:
        apart.close()


@pytest.mark.parametrize("n_xcd", [1, 4, 8])
@pytest.mark.parametrize("nMacM,nMacN", [(1, 1), (28, 8), (29, 8), (5, 57), (33, 9), (4, 505), (32, 64), (29, 63), (17, 97)])
def test_schedule_of_few_super_tiles_deals_every_macro_tile_once(nMacM, nMacN, n_xcd):
    """At most 64 super tiles of C are scheduled a super tile a lane: below, at and above the number of XCDs, up to
    64 and one more, ragged in either direction, some of them with nothing kept.  Macro tiles and computing ones per XCD are those of
    the greedy deal, and C, NaN before, is the product (whole numbers: every sum is exact)."""
    import torch
    import cuspamm_amd as sp
    tile, rng = 128, np.random.default_rng(nMacM * 1000 + nMacN)
    M, K, N = nMacM * 256 - 128, 16 * tile, nMacN * 256 - 128
    A = torch.from_numpy(rng.integers(-2, 3, (M, K)).astype(np.float32)).cuda()
    B = torch.from_numpy(rng.integers(-2, 3, (K, N)).astype(np.float32)).cuda()
    for i in range(0, M, tile):                          # lists of different lengths, groups of rows without any
        A[i:i + tile, (0 if i // 1024 % 3 == 1 else rng.integers(0, 17)) * tile:] = 0.0
    B[:, -N // 4:] = 0.0
    other = sp.SpammContext(0)
    try:
        other.set_option(sp.OPT_NUM_XCD, n_xcd)
        other.set_option(sp.OPT_GEMM_SHAPE, 1)
        C = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        other.multiply(A, B, tile, 1.0, C=C)
        counts, sched = other.get_macro_counts()
    finally:
        other.close()
    assert torch.equal(C, A @ B)
    supers = [counts[i:i + 4, j:j + 8, 0] for i in range(0, nMacM, 4) for j in range(0, nMacN, 8)]
    rounds, want = -(-len(supers) // n_xcd), [[0, 0, 0, 0] for _ in range(n_xcd)]      # length, super tiles, computing, all
    if len(supers) < n_xcd:
        chunk = -(-counts[..., 0].size // n_xcd)
        for x in range(n_xcd):
            part = counts[..., 0].reshape(-1)[x * chunk:(x + 1) * chunk]
            want[x][2:] = [np.count_nonzero(part), part.size]
    else:
        for s in sorted(supers, key=lambda s: -int(s.sum())):
            room = [x for x in range(n_xcd) if want[x][1] < rounds]
            x = min(room, key=lambda x: (want[x][0], x)) if s.any() else room[0]
            for n, v in enumerate((int(s.sum()), 1, np.count_nonzero(s), s.size)):
                want[x][n] += v
    assert [list(v) for v in zip(sched[:n_xcd], sched[8:8 + n_xcd])] == [w[2:] for w in want]


def test_schedule_of_the_longest_lists_on_one_xcd(ctx):
    """One XCD takes every super tile of a band, and the lengths dealt to it so far are part of the key it is chosen by:
    lists of 65535 k tiles bring that sum to 2^28 - 1 before the last super tile is dealt (times 8, plus the XCD's number:
    more than 31 bits).  Every macro tile must be in the sequence."""
    import cuspamm_amd as sp
    nbM, nbK, nbN, tile = 14 * 8, 65535, 16 * 16, 128            # 14 x 16 super tiles of 8 x 16 output tiles
    nA = np.zeros((nbM, nbK), np.float32)
    nB = np.ones((nbK, nbN), np.float32)
    nA[:64] = 1.0                                                # 128 super tiles whose 32 lists hold every k: 268431360 in all,
    nA[64:66] = 0.5
    nB[:4095, 0] = 2.0                                           # one with a single list of 4095,
    nB[:5, 16] = 2.0                                             # and one with a single list of 5
    other = sp.SpammContext(0)
    try:
        other.set_option(sp.OPT_NUM_XCD, 1)
        other.set_normmaps(nA, nB, tile)
        other.gate(1.0)
        counts, sched = other.get_macro_counts()
        work = counts[..., 0]
        assert work[:32].min() == 65535 and work[32:].sum() == 4095 + 5
        assert sched[0] == np.count_nonzero(work) == 32 * 128 + 2
        assert sched[8] == work.size
    finally:
        other.close()


@pytest.mark.parametrize("ring", [3, 5])
def test_other_staging_rings_give_the_same_product(orc, ctx, ring):
    """The GEMM's ring of LDS stages is four deep by default; three and five walk the same lists.  Lists shorter than
    the ring, empty ones, an odd number of entries kept by all tiles (tile 32: one stage each), ragged edges of C."""
    import torch
    import cuspamm_amd as sp
    other = sp.SpammContext(0)
    other.set_option(sp.OPT_GEMM_RING, ring)
    other.set_option(sp.OPT_GEMM_SHAPE, 1)
    ctx.set_option(sp.OPT_GEMM_SHAPE, 1)
    try:
        for (M, K, N), tile, lam, ratio in [((256, 32, 256), 32, 0.0, 1.0), ((256, 96, 512), 32, 0.0, 1.0), ((512, 224, 256), 32, 0.0, 1.0),
                                            ((1280, 512, 768), 32, 0.01, 0.5), ((96, 64, 160), 32, 0.0, 1.0),
                                            ((2304, 1024, 4352), 64, 0.004, 0.3), ((320, 64, 448), 64, 0.0, 1.0),
                                            ((640, 4096, 896), 128, 0.001, 0.1), ((128, 128, 128), 128, 0.0, 1.0)]:
            tab = orc.decay_table("exp", max(M, K, N), lam)
            dA, dB = _dev(orc.fill_decay(M, K, tab, 1)), _dev(orc.fill_decay(K, N, tab, 2))
            ctx.normmap_f32(1, dB, tile)
            ctx.normmap_f32(0, dA, tile)
            tau = 0.0 if ratio == 1.0 else ctx.tau_for_ratio(ratio)[0]
            want = ctx.multiply(dA, dB, tile, tau)
            got = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
            other.multiply(dA, dB, tile, tau, C=got)
            assert torch.equal(got, want), (M, K, N, tile)
            assert np.array_equal(other.get_mask(), ctx.get_mask())
        tab = orc.decay_table("exp", 2048, 0.003)
        _check(orc, other, orc.fill_decay(384, 2048, tab, 3), orc.fill_decay(2048, 320, tab, 4), 32, 0.05)
    finally:
        ctx.set_option(sp.OPT_GEMM_SHAPE, 0)
        other.close()


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("tile", [32, 64, 128])
def test_passes_over_small_inputs_end_strips_anywhere(orc, ctx, tile, half):
    """The passes of small inputs, whose strips of up to eight tiles end at the last column or before it: each operand by itself, both in
    one launch and A = B, copies and norm maps bit for bit, with tiles of zeros, subnormals and values from 2^-24 to 2^15; and a tau-aware
    call beside a plain one."""
    import torch
    rng = np.random.default_rng(tile + half)
    kind = torch.float16 if half else torch.float32

    def operand(rows, cols):
        x = (rng.uniform(-1.0, 1.0, (rows, cols)) * 2.0 ** rng.integers(-24, 16, (rows, cols))).astype(np.float32)
        x[:tile, cols - tile:] = 0.0
        x[rows - tile:, :tile] *= rng.random((tile, tile)) < 0.01
        return torch.from_numpy(x).cuda().to(kind)

    def same(role, X):
        bits = X.half().cpu().numpy().view(np.uint16)
        assert np.array_equal(ctx.get_fp16(role), bits)
        assert np.array_equal(ctx.get_normmap(role).view(np.uint32), orc.normmap(bits, tile, role).view(np.uint32))

    alone = ctx.normmap_f16 if half else ctx.normmap_f32
    for m, k, n in ((1, 1, 1), (1, 2, 3), (3, 5, 7), (2, 8, 9), (9, 16, 4), (5, 17, 15)):
        A, B = operand(m * tile, k * tile), operand(k * tile, n * tile)
        alone(1, B, tile)
        alone(0, A, tile)
        same(0, A)
        same(1, B)
        want = ctx.multiply(A, B, tile, 0.5)
        same(0, A)
        same(1, B)
        got = ctx.multiply(A, B, tile, 0.5, prune=True)
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(want)) and torch.equal(got.isnan(), want.isnan())
    for n in (1, 3, 8, 9):
        A = operand(n * tile, n * tile)
        ctx.multiply(A, A, tile, 0.5, a_eq_b=True)
        same(0, A)
        same(1, A)


@pytest.mark.parametrize("tile,half,n", [(32, False, 2912), (32, True, 4128), (64, False, 2944), (64, False, 4160), (64, True, 4160)])
def test_passes_over_inputs_beyond_the_cache_line(orc, ctx, tile, half, n):
    """The same beyond 32 MiB an operand, where rows are streamed past the caches: ragged strips, each operand by itself, both in one
    launch, A = B, and a tau-aware call beside a plain one."""
    import torch
    kind = torch.float16 if half else torch.float32
    m = n + tile
    tab = orc.decay_table("exp", m, 0.01)
    A = torch.empty((m, n), dtype=torch.float32, device="cuda")
    B = torch.empty((n, m), dtype=torch.float32, device="cuda")
    ctx.fill_decay(A, tab, 1)
    ctx.fill_decay(B, tab, 2)
    A, B = A.to(kind), B.to(kind)

    def same(role, X):
        bits = X.half().cpu().numpy().view(np.uint16)
        assert np.array_equal(ctx.get_fp16(role), bits)
        assert np.array_equal(ctx.get_normmap(role).view(np.uint32), orc.normmap(bits, tile, role).view(np.uint32))

    alone = ctx.normmap_f16 if half else ctx.normmap_f32
    alone(1, B, tile)
    alone(0, A, tile)
    same(0, A)
    same(1, B)
    tau = ctx.tau_for_ratio(0.05)[0]
    want = ctx.multiply(A, B, tile, tau)
    same(0, A)
    same(1, B)
    assert torch.equal(ctx.multiply(A, B, tile, tau, prune=True), want)
    X = A[:n].contiguous()
    ctx.multiply(X, X, tile, tau, a_eq_b=True)
    same(0, X)
    same(1, X)


@pytest.mark.parametrize("tile,half,M,K,N", [(32, True, 288, 352, 544), (64, True, 320, 192, 448), (128, True, 384, 256, 640),      # one launch
                                             (32, True, 4064, 4128, 1056), (64, True, 4032, 4160, 1088), (64, True, 4096, 4096, 576),
                                             (128, True, 4224, 4096, 1152),
                                             (32, False, 288, 352, 544), (64, False, 320, 192, 448), (128, False, 384, 256, 640),
                                             (32, False, 3104, 2848, 1056), (64, False, 3136, 2816, 1088), (64, False, 2816, 8192, 2112)])
def test_matrices_begin_anywhere(ctx, tile, half, M, K, N):
    """Operands that begin at any element of a buffer, halves between two 32-bit words among them, and C at any float: bit for bit as where all
    begin at 256 bytes, in passes of their own, both in one launch, A = B, tau-aware, small and beyond 32 MiB."""
    import torch
    tab = np.exp(-0.005 * np.arange(max(M, K, N))).astype(np.float32)

    def filled(rows, cols, seed):
        X = torch.empty((rows, cols), dtype=torch.float32, device="cuda")
        ctx.fill_decay(X, tab, seed)
        return X.half() if half else X

    def at(X, offset):
        buffer = torch.full((X.numel() + 8,), float("nan"), dtype=X.dtype, device="cuda")
        view = buffer[offset:offset + X.numel()].view(X.shape)
        view.copy_(X)
        return view, buffer

    def state(*roles):
        return [ctx.get_normmap(r).view(np.uint32) for r in roles] + [ctx.get_fp16(r) for r in roles]

    def same(got, want):
        assert all(np.array_equal(g, w) for g, w in zip(got, want))

    A, B = filled(M, K, 1), filled(K, N, 2)
    alone = ctx.normmap_f16 if half else ctx.normmap_f32
    alone(1, B, tile)
    alone(0, A, tile)
    tau = ctx.tau_for_ratio(0.2)[0]
    C = ctx.multiply(A, B, tile, tau)
    want, mask = state(0, 1), ctx.get_mask()
    n = min(M, K)
    S = A[:n, :n].contiguous()
    square = ctx.multiply(S, S, tile, tau, a_eq_b=True)
    want_square = state(0, 1)
    for a, b, c in ((1, 0, 0), (0, 1, 1), (3, 2, 3), (2, 5, 0)):
        (Av, _), (Bv, _), (Cv, buffer) = at(A, a), at(B, b), at(torch.empty_like(C), c)
        assert Av.data_ptr() % 16 == (a * A.element_size()) % 16 and Av.is_contiguous()
        alone(1, Bv, tile)
        alone(0, Av, tile)
        same(state(0, 1), want)
        ctx.multiply(Av, Bv, tile, tau, C=Cv)
        same(state(0, 1), want)
        assert torch.equal(Cv, C) and np.array_equal(ctx.get_mask(), mask)
        assert buffer[:c].isnan().all() and buffer[c + C.numel():].isnan().all()
        Cv.fill_(float("nan"))
        ctx.multiply(Av, Bv, tile, tau, C=Cv, prune=True)
        assert torch.equal(Cv, C) and np.array_equal(ctx.get_mask(), mask)
        if not half and max(M * K, K * N) * 2 <= 16 << 20:
            Cv.fill_(float("nan"))
            ctx.multiply_noalloc(Av, Bv, tile, tau, Cv)
            assert torch.equal(Cv, C)
        Sv, _ = at(S, a)
        assert torch.equal(ctx.multiply(Sv, Sv, tile, tau, a_eq_b=True), square)
        same(state(0, 1), want_square)
