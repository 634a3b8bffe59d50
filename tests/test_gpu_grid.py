"""Pairs cut into a grid of tiles and merged on both sides, row pads of the
32-bit chain and the budget fallback, against the oracle bit for bit."""
import numpy as np
import pytest

import lcs_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with lcs_amd.Context(0) as c:
        yield c


def check(ctx, a, b, sched=None):
    h, v, score = ctx.comb(a, b, sched)
    ho, vo = oracle.comb(a, b, order="mt")
    assert np.array_equal(h, ho) and np.array_equal(v, vo)
    assert score == int((vo < a.size).sum())


def pair(seed, m, n, alphabet):
    a = lcs_amd.gen_uniform(seed, m, alphabet)
    return a, lcs_amd.gen_mutate(seed + 1, a, alphabet, 0.1, 0.02, n)


# sizes on both sides of the first cut (2^26 cells), uneven last tiles, tall,
# wide and odd grids
@pytest.mark.parametrize("m,n,alphabet", [(8191, 8192, 4), (8192, 8193, 4), (9001, 7777, 20), (4099, 40001, 4),
                                          (40001, 4099, 26), (2500, 65537, 4), (16411, 30011, 300),
                                          (50021, 33333, 4)])
def test_cut_pairs_match_oracle(ctx, m, n, alphabet):
    check(ctx, *pair(m, m, n, alphabet))


@pytest.mark.parametrize("symbols", [[-1, -2, 7, 1 << 20], list(range(-24, 0)), list(range(-23, 0)) + [1 << 30],
                                     [-24, -25, 300]])
@pytest.mark.parametrize("tm", [1, 4, 16])
def test_partial_bands_of_wide_symbols(ctx, symbols, tm):
    # the last band's rows are padded with one of -1 .. -24 that b does not
    # hold, and masked when b holds them all
    rng = np.random.default_rng(tm)
    for m, n in ((1, 40), (64 * tm + 1, 333), (64 * tm * 2 - 1, 1000)):
        a, b = (rng.choice(np.array(symbols, np.int32), x) for x in (m, n))
        check(ctx, a, b, lcs_amd.schedule(tm, 1, lcs_amd.VARIANT_CHAIN, 1))


def test_small_budget_falls_back_to_one_tile():
    a, b = pair(3, 9000, 9000, 4)
    with lcs_amd.Context(0, hbm_budget=2 << 20) as c:
        check(c, a, b)
        assert c.memory()[0] <= 2 << 20


def test_plans_agree_with_one_tile(ctx):
    for m, n in ((131072, 9000), (9000, 131072), (70001, 70001)):
        a, b = pair(m, m, n, 4)
        whole = ctx.comb(a, b, lcs_amd.schedule(4, 1, lcs_amd.VARIANT_CHAIN, 1))
        cut = ctx.comb(a, b)
        assert np.array_equal(whole[0], cut[0]) and np.array_equal(whole[1], cut[1])


@pytest.mark.parametrize("m,n,alphabet", [(1, 16384, 2), (5, 40001, 300), (64, 100003, 4), (300, 60000, 256),
                                          (1024, 16385, 40000), (4000, 16400, 20)])
def test_wide_short_pairs_match_oracle(ctx, m, n, alphabet):
    # below the cells from which a pair is cut both ways: columns only
    check(ctx, *pair(m + n, m, n, alphabet))
