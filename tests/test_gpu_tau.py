"""Device-side tau selection against the host checker (tool.cu:438-490 semantics)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _maps(rng, nbM, nbK, nbN, zero_frac=0.0):
    nA = np.abs(rng.normal(size=(nbM, nbK))).astype(np.float32) * 10 ** rng.uniform(-3, 1, size=(nbM, nbK)).astype(np.float32)
    nB = np.abs(rng.normal(size=(nbK, nbN))).astype(np.float32)
    if zero_frac:
        nA[rng.random(nA.shape) < zero_frac] = 0
    return nA.astype(np.float32), nB.astype(np.float32)


@pytest.mark.parametrize("shape", [(8, 32, 8), (5, 70, 3), (33, 130, 17), (64, 64, 64), (1, 1, 1)])
def test_order_statistic_matches_checker(orc, ctx, shape):
    rng = np.random.default_rng(sum(shape))
    nA, nB = _maps(rng, *shape)
    ctx.set_normmaps(nA, nB, 64)
    for ratio in (0.0, 0.01, 0.1, 0.5, 0.75, 0.999, 1.0):
        tau_g, ach_g = ctx.tau_for_ratio(ratio)
        tau_o, ach_o = orc.tau_for_ratio(nA, nB, ratio)
        assert np.float32(tau_g) == np.float32(tau_o), (ratio, tau_g, tau_o)
        assert ach_g == ach_o
        # and the gate at that tau keeps exactly that many products
        ctx.gate(tau_g)
        assert ctx.get_stats().kept_products == round(ach_g * nA.shape[0] * nA.shape[1] * nB.shape[1])


def test_zero_tail_and_all_zero(orc, ctx):
    rng = np.random.default_rng(1)
    nA, nB = _maps(rng, 16, 48, 16, zero_frac=0.8)
    ctx.set_normmaps(nA, nB, 32)
    for ratio in (0.1, 0.5, 0.9):                              # 0.5 and 0.9 are unreachable with tau > 0
        tau_g, ach_g = ctx.tau_for_ratio(ratio)
        tau_o, ach_o = orc.tau_for_ratio(nA, nB, ratio)
        assert np.float32(tau_g) == np.float32(tau_o) and ach_g == ach_o
        assert tau_g > 0
    ctx.set_normmaps(np.zeros((4, 4), np.float32), np.ones((4, 4), np.float32), 32)
    assert ctx.tau_for_ratio(0.3) == (0.0, 1.0)


def test_count_kept(ctx):
    rng = np.random.default_rng(2)
    nA, nB = _maps(rng, 20, 100, 12)
    ctx.set_normmaps(nA, nB, 64)
    p = (nA[:, None, :] * nB.T[None, :, :]).astype(np.float64)
    for thr in (0.0, 1e-3, 0.5, 7.0):
        cnt, sm = ctx.count_kept(thr)
        assert cnt == int((p >= thr).sum())
        assert abs(sm - p.sum()) <= 1e-9 * p.sum()


def test_reference_bisection(orc, ctx):
    rng = np.random.default_rng(3)
    for shape in [(8, 32, 8), (32, 64, 32)]:
        nA, nB = _maps(rng, *shape)
        ctx.set_normmaps(nA, nB, 32)
        for expected in (0.75, 0.3):
            tau_g, ach_g = ctx.tune_bisect(expected, 0.01, 20)
            tau_o, ach_o = orc.tune_bisect(nA, nB, expected, 0.01, 20)
            assert abs(tau_g - tau_o) <= 1e-6 * abs(tau_o)      # the mean product is summed in another order
            assert abs(ach_g - ach_o) <= 2.0 / (shape[0] * shape[1] * shape[2])
            assert abs(ach_g - expected) < 0.01


def test_bisection_iterates_match_the_hand_worked_sequence(ctx):
    # the sequences worked by hand from tool.cu:445-486 (products 1, 2, 3, 4; all sums exact)
    from test_oracle_gate import BISECT_HAND
    ctx.set_normmaps(np.array([[1.0, 2.0, 3.0, 4.0]], dtype=np.float32), np.ones((4, 1), dtype=np.float32), 32)
    for expected, seq in BISECT_HAND.items():
        for rounds, want in enumerate(seq, start=1):
            assert ctx.tune_bisect(expected, 0.01, rounds) == want, (expected, rounds)
    assert ctx.tune_bisect(0.25, 0.01, 20) == (3.75, 0.25)
    assert ctx.tune_bisect(0.75, 0.01, 20) == (1.25, 0.75)


def test_dropped_bound_hand_worked(ctx):
    # per output tile the dropped products sum to 7, 10, 4, 8 at tau = 10 and to 7, 2, 4, 0 at
    # tau = 8 (a product equal to tau is kept)
    nA = np.array([[1, 2, 3], [4, 5, 6]], dtype=np.float32)
    nB = np.array([[1, 2], [3, 4], [5, 6]], dtype=np.float32)
    ctx.set_normmaps(nA, nB, 32)
    assert ctx.dropped_bound(10.0) == pytest.approx(np.sqrt(229.0), rel=1e-14)
    assert ctx.dropped_bound(8.0) == pytest.approx(np.sqrt(69.0), rel=1e-14)
    assert ctx.dropped_bound(0.0) == 0.0


def test_full_size_selection(orc, ctx):
    import torch
    N, tile = 16384, 64
    tab = orc.decay_table("exp", N, 0.003)
    dA = torch.empty((N, N), dtype=torch.float32, device="cuda")
    dB = torch.empty((N, N), dtype=torch.float32, device="cuda")
    ctx.fill_decay(dA, tab, 1)
    ctx.fill_decay(dB, tab, 2)
    ctx.normmap_f32(1, dB, tile)
    ctx.normmap_f32(0, dA, tile)
    tau_g, ach_g = ctx.tau_for_ratio(0.10)
    tau_o, ach_o = orc.tau_for_ratio(ctx.get_normmap(0), ctx.get_normmap(1), 0.10)
    assert np.float32(tau_g) == np.float32(tau_o) and ach_g == ach_o
    assert abs(ach_g - 0.10) < 1e-4


@pytest.mark.parametrize("shape", [(1, 63, 16), (3, 64, 17), (2, 65, 15), (129, 65, 33), (40, 1, 300), (1, 1000, 1)])
def test_selection_at_the_edges_of_its_work_units(orc, ctx, shape):
    # units of 16 columns x 64 k: remainders of both, one product more or less; ties, zeros and the wanted rank
    # at the ends of a digit's bin.  tau and kept counts are whole-number results: exact
    rng = np.random.default_rng(sum(shape))
    nA, nB = _maps(rng, *shape, zero_frac=0.3)
    total = shape[0] * shape[1] * shape[2]
    for a, b in ((nA, nB), (np.full_like(nA, 3.0), np.full_like(nB, 0.5)), (np.round(nA * 4), np.round(nB * 4))):
        ctx.set_normmaps(a, b, 32)
        for ratio in (1.0 / total, 0.37, 0.5, 1.0 - 1.0 / total, 1.0):
            got, want = ctx.tau_for_ratio(ratio), orc.tau_for_ratio(a, b, ratio)
            assert np.float32(got[0]) == np.float32(want[0]) and got[1] == want[1], (ratio, got, want)


@pytest.mark.parametrize("rounds", [1, 2, 4, 5, 6, 9, 20, 21, 22, 45])
def test_bisection_stops_at_any_round(orc, ctx, rounds):
    # several rounds per launch, twenty per wait: remainders of both, on a target that is never met (the kept
    # fractions of 6 products are sixths), so that exactly `rounds` rounds run; sums of these values are exact
    nA, nB = np.array([[1.0, 2.0, 4.0], [0.5, 8.0, 16.0]], np.float32), np.ones((3, 1), np.float32)
    ctx.set_normmaps(nA, nB, 32)
    got, want = ctx.tune_bisect(0.4, 0.01, rounds), orc.tune_bisect(nA, nB, 0.4, 0.01, rounds)
    assert np.float32(got[0]) == np.float32(want[0]) and got[1] == want[1]


@pytest.mark.parametrize("shape", [(1, 8192, 1), (1, 8193, 1), (3, 1024, 8), (7, 3511, 1), (1, 24577, 1)])
def test_selection_at_the_edges_of_what_one_workgroup_holds(orc, ctx, shape):
    # 8 and 24 products per thread of 1024, and one more than each: exact, as above
    rng = np.random.default_rng(sum(shape))
    nA, nB = _maps(rng, *shape, zero_frac=0.3)
    nA[0, 0] = np.nan                                          # (a NaN product is never kept, and counts as zero)
    total = shape[0] * shape[1] * shape[2]
    clean = np.where(np.isnan(nA), 0, nA).astype(np.float32)
    for a, b, oa in ((nA, nB, clean), (np.round(clean * 4), np.round(nB * 4), np.round(clean * 4))):
        ctx.set_normmaps(a, b, 32)
        for ratio in (1.0 / total, 0.37, 0.6, 1.0):
            got, want = ctx.tau_for_ratio(ratio), orc.tau_for_ratio(oa, b, ratio)
            assert np.float32(got[0]) == np.float32(want[0]) and got[1] == want[1], (ratio, got, want)


@pytest.mark.parametrize("repeat", [1, 1365, 1366, 4096, 4097])
@pytest.mark.parametrize("rounds", [1, 5, 6, 20, 22])
def test_bisection_stops_at_any_round_with_many_products(orc, ctx, repeat, rounds):
    # the six products above, `repeat` times: 8190, 8196, 24576 products of one workgroup, 24582 of many.
    # Sums of these values are exact in any order
    nA = np.tile(np.array([[1.0, 2.0, 4.0], [0.5, 8.0, 16.0]], np.float32), (1, repeat))
    nB = np.ones((3 * repeat, 1), np.float32)
    ctx.set_normmaps(nA, nB, 32)
    got, want = ctx.tune_bisect(0.4, 0.01, rounds), orc.tune_bisect(nA, nB, 0.4, 0.01, rounds)
    assert np.float32(got[0]) == np.float32(want[0]) and got[1] == want[1]


@pytest.mark.parametrize("repeat", [1, 4097])
@pytest.mark.parametrize("expected", [0.4, 2.0])
def test_bisection_without_a_limit_ends_where_its_thresholds_do(orc, ctx, repeat, expected):
    # a target that is never met and no limit worth the name: doubles have no threshold left between two kept
    # fractions after some 60 rounds, or below the smallest product after 1100, and further rounds change nothing
    nA = np.tile(np.array([[1.0, 2.0, 4.0], [0.5, 8.0, 16.0]], np.float32), (1, repeat))
    nB = np.ones((3 * repeat, 1), np.float32)
    ctx.set_normmaps(nA, nB, 32)
    got, want = ctx.tune_bisect(expected, 0.01, 2 ** 31 - 1), orc.tune_bisect(nA, nB, expected, 0.01, 1200)
    assert np.float32(got[0]) == np.float32(want[0]) and got[1] == want[1]


@pytest.mark.parametrize("repeat", [1, 1366, 4097])
@pytest.mark.parametrize("rounds", [2, 5, 20])
def test_bisection_over_uploaded_maps_with_negative_values(orc, ctx, repeat, rounds):
    # hand-built maps may hold any value: the mean product and with it the thresholds are negative here, and the
    # lanes without a product must count for none of them.  Sums of these values are exact in any order
    nA = np.tile(np.array([[-1.0, -2.0, 4.0], [-0.5, -8.0, -16.0]], np.float32), (1, repeat))
    nB = np.ones((3 * repeat, 1), np.float32)
    ctx.set_normmaps(nA, nB, 32)
    for expected in (0.4, 0.9):
        got, want = ctx.tune_bisect(expected, 0.01, rounds), orc.tune_bisect(nA, nB, expected, 0.01, rounds)
        assert np.float32(got[0]) == np.float32(want[0]) and got[1] == want[1], (expected, got, want)


def test_results_on_one_stream_after_another(orc):
    # a result is handed out before its stream is idle: the next call, on another stream, finds the workspace at rest
    import torch
    import cuspamm_amd as sp
    rng = np.random.default_rng(5)
    nA, nB = _maps(rng, 48, 70, 40, zero_frac=0.2)
    ratios = (0.02, 0.3, 0.7)
    want = [orc.tau_for_ratio(nA, nB, r) for r in ratios]
    prods = nA[:, None, :].astype(np.float64) * nB.T[None].astype(np.float64)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    c = sp.SpammContext(0)
    try:
        c.set_normmaps(nA, nB, 32)
        for rep in range(24):
            c.set_stream(streams[rep % 2].cuda_stream)
            r = rep % 3
            got = c.tau_for_ratio(ratios[r])
            assert np.float32(got[0]) == np.float32(want[r][0]) and got[1] == want[r][1], rep
            if rep % 4 == 3:
                c.set_stream(streams[(rep + 1) % 2].cuda_stream)
                assert c.count_kept(0.0)[0] == nA.shape[0] * nA.shape[1] * nB.shape[1]
                # sums of 134400 fp64 terms in another order: below 134400 * 2^-53 = 1.5e-11 of the sum of squares
                assert c.dropped_bound(float("inf")) == pytest.approx(np.sqrt((prods.sum(axis=2) ** 2).sum()), rel=1.5e-11)
    finally:
        c.close()


@pytest.mark.parametrize("shape", [(40, 130, 23), (64, 64, 64), (1, 40000, 1), (300, 1, 301)])
@pytest.mark.parametrize("rounds", [2, 11, 12, 21, 22, 32])
def test_bisection_by_a_search_tree(orc, ctx, shape, rounds):
    # ten rounds per launch, twenty per wait, on one stream and then another: remainders of the work units, ties,
    # zeros, many octaves, and kept fractions at the ends.  Products of small whole numbers (times a power of two): their
    # sums are exact in any order, so thresholds and fractions are those of the checker bit for bit
    import torch
    rng = np.random.default_rng(sum(shape) + rounds)
    nA = rng.integers(0, 64, size=shape[:2]).astype(np.float32)
    nB = (2.0 ** rng.integers(-6, 7, size=shape[1:])).astype(np.float32)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for at, expected in enumerate((0.75, 0.2, 0.003, 0.999, 2.0)):
        ctx.set_stream(streams[at % 2].cuda_stream)
        ctx.set_normmaps(nA, nB, 32)
        for tol in (0.01, 1e-7):
            got, want = ctx.tune_bisect(expected, tol, rounds), orc.tune_bisect(nA, nB, expected, tol, rounds)
            assert np.float32(got[0]) == np.float32(want[0]) and got[1] == want[1], (expected, tol, got, want)
    ctx.set_stream(None)


@pytest.mark.parametrize("workgroups", [47, 48, 49, 63, 65, 256])
def test_counts_of_few_and_many_workgroups(ctx, workgroups):
    """Workgroups of a pass hand their part to the one that ends last, found by one ticket (up to 48) or by groups' tickets:
    every product is counted once, and again in the next call (16 products of a norm map row in 64 k each per wave)."""
    rng = np.random.default_rng(workgroups)
    nA = rng.random((16 * workgroups, 64), dtype=np.float32)
    nB = rng.random((64, 16), dtype=np.float32)
    p = nA[:, None, :] * np.ascontiguousarray(nB.T)[None]
    ordered = np.sort(p.ravel())
    ctx.set_normmaps(nA, nB, 32)
    for _ in range(2):
        for thr in (0.0, 0.25, 0.9):
            assert ctx.count_kept(thr)[0] == np.count_nonzero(p.astype(np.float64) >= thr)
        tau, achieved = ctx.tau_for_ratio(0.3)
        assert np.float32(tau) == ordered[p.size - int(np.ceil(0.3 * p.size))]
        assert achieved == np.count_nonzero(p >= np.float32(tau)) / p.size
        tau, achieved = ctx.tune_bisect(0.5, 0.01, 20)
        assert abs(achieved - 0.5) < 0.01 and abs(np.count_nonzero(p >= np.float32(tau)) / p.size - achieved) < 1e-6
        assert ctx.dropped_bound(0.5) == pytest.approx(np.sqrt((np.where(p < 0.5, p.astype(np.float64), 0.0).sum(axis=2) ** 2).sum()), rel=1e-6)


@pytest.mark.parametrize("nbK", [1023, 1025])
def test_selection_of_products_that_fit_32_bits_and_more(ctx, nbK):
    """Below 2^32 products two bins share a word of the histogram.  Products of row i are all i + 1: what a kept fraction
    selects is known."""
    nbM = nbN = 2048
    nA = np.repeat(np.arange(1, nbM + 1, dtype=np.float32)[:, None], nbK, axis=1)
    ctx.set_normmaps(nA, np.ones((nbK, nbN), np.float32), 32)
    per_row, total = nbK * nbN, nbM * nbK * nbN
    for ratio in (0.0, 1e-4, 0.3, 0.999, 1.0):
        want = min(max(1, int(np.ceil(ratio * float(total)))), total)
        row = nbM - (want - 1) // per_row
        tau, achieved = ctx.tau_for_ratio(ratio)
        assert tau == row and achieved == (nbM - row + 1) * per_row / total


def test_bisection_of_more_products_than_workgroups_count(orc, ctx):
    """Beyond 2^38 products a pass has more workgroups than the chip runs at once.  Products of row i are all i + 1, 2^24 of
    each: kept fractions and the mean are those of one product a row, whose bisection the checker has."""
    nbM, nbK, nbN = 16640, 1024, 16384
    rows = np.arange(1, nbM + 1, dtype=np.float32)[:, None]
    ctx.set_normmaps(np.repeat(rows, nbK, axis=1), np.ones((nbK, nbN), np.float32), 32)
    for expected in (0.5, 0.003):
        got, want = ctx.tune_bisect(expected, 1e-4, 20), orc.tune_bisect(rows, np.ones((1, 1), np.float32), expected, 1e-4, 20)
        assert np.float32(got[0]) == np.float32(want[0]) and got[1] == want[1]


@pytest.mark.parametrize("shape", [(65535, 1, 4096), (65535, 1, 4112), (3, 200, 33), (2, 64 * 130 + 1, 5)])
def test_steps_by_reciprocals_and_by_divisions_visit_every_product(ctx, shape):
    """Where a step's number times the divisor leaves 32 bits (65535 x 257 groups of columns) the steps are divided for; the shapes beside
    it go by reciprocals.  Norms are powers of two, so products are too, and their distribution is the sum of the exponents'."""
    nbM, nbK, nbN = shape
    rng = np.random.default_rng(nbM + nbN)
    ea, eb = rng.integers(0, 8, (nbM, nbK)), rng.integers(0, 8, (nbK, nbN))
    ctx.set_normmaps((2.0 ** -ea).astype(np.float32), (2.0 ** -eb).astype(np.float32), 32)
    having = np.zeros(15, dtype=np.int64)                        # products of 2^-e
    for x in range(8):
        for y in range(8):
            having[x + y] += int(((ea == x).sum(axis=0) * (eb == y).sum(axis=1)).sum())
    upto = np.cumsum(having)
    assert upto[-1] == nbM * nbK * nbN
    for e in (0, 3, 7, 14):
        cnt, sm = ctx.count_kept(2.0 ** -e)
        assert cnt == upto[e]
        assert abs(sm - (having * 2.0 ** -np.arange(15.0)).sum()) <= 1e-9 * sm
    for ratio in (0.01, 0.3, 0.9):
        e = int(np.searchsorted(upto, np.ceil(ratio * upto[-1])))
        tau, achieved = ctx.tau_for_ratio(ratio)
        assert tau == 2.0 ** -e and achieved == upto[e] / upto[-1]
    tau, achieved = ctx.tune_bisect(0.5, 0.2, 20)
    assert achieved == np.float32(upto[int(np.floor(-np.log2(tau)))]) / np.float32(upto[-1])
